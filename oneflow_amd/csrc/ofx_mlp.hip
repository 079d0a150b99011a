// ofx_mlp.hip -- the warm-start predictor: a BF16 multilayer perceptron
// (inputs 9 -> 5 hidden layers of 256 with SiLU -> 5 outputs) trained and
// evaluated with hand-written MFMA kernels on the GPU.  No counterpart in the
// reference: it predicts a starting flow field, and the solver then iterates
// from it to the same tolerance as from freestream.
//
// Numerics: weights are kept in FP32 (Adam master copy) and used in BF16;
// activations between layers are BF16; every product is accumulated in FP32
// by v_mfma_f32_16x16x32_bf16.  Pre-activations are kept in FP32 for the
// backward pass.
//
// Layout: activations row-major [samples][features]; weights [in][out]
// row-major, with a transposed bf16 copy [out][in] for the forward products
// (the GEMM reads both operands along k).  Feature counts are padded: input 9 -> 16, output 5 -> 64 (the
// padding weights are zero and stay zero: their gradients are exactly zero);
// the sample count is padded to a multiple of 64 with zero rows that carry no
// loss.
#include "ofx_common.h"

#include <condition_variable>
#include <mutex>
#include <thread>

namespace ofx {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
typedef float v8f __attribute__((ext_vector_type(8)));
typedef uint16_t v8us __attribute__((ext_vector_type(8)));
typedef uint16_t bf16;

constexpr int NIN = 9, NIN_P = 16, NHID = 256, NLAYER = 6, NOUT = 5, NOUT_P = 64;
constexpr int MLP_MAXN = 1 << 20;  // samples per call
constexpr int SPLITK_CHUNK = 1024;

__device__ __forceinline__ bf16 f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
    return (bf16)(u >> 16);
}
__device__ __forceinline__ float bf2f(bf16 h) { return __uint_as_float(((uint32_t)h) << 16); }
// SiLU and its derivative with the hardware reciprocal (v_rcp_f32, 1 ulp)
// instead of a correctly rounded division: the epilogues evaluate one per
// output element, and a division is ten instructions against one.  The
// values feed BF16 activations, whose rounding is 2^-9 relative.
__device__ __forceinline__ float sigm(float z) { return __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }
__device__ __forceinline__ float silu(float z) { return z * sigm(z); }
__device__ __forceinline__ float dsilu(float z) {
    float s = sigm(z);
    return s * (1.0f + z * (1.0f - s));
}

enum { EPI_BIAS_SILU = 0, EPI_BIAS = 1 };

// C[M x N] = A[M x K] Bt[N x K]^T: both operands bf16 with k contiguous
// (row strides lda, ldb), so every global and LDS access moves 8 elements
// (16 bytes) at a time.  BM x BN block tile (64 or 128 each; M and N
// multiples of them); K a multiple of 16 (an 8-element vector at or past its end is
// zero-filled, so K = 16 runs through the 32-deep MFMA with zero products
// added).  256 threads: wave w owns rows (BM/2)*(w>>1).. and columns
// (BN/2)*(w&1).. as (BM/32) x (BN/32) tiles of gfx950's
// v_mfma_f32_16x16x32_bf16.  MFMA operands: lane l supplies A[l%16][8*(l/16)
// + 0..7] and Bt[l%16][8*(l/16) + 0..7] and receives D[4*(l/16)+r][l%16],
// r = 0..3.  K advances KC at a time through LDS (one barrier pair per KC/32
// MFMA steps); the next chunk's global loads are issued into registers before
// the current chunk's MFMAs, so their latency overlaps the arithmetic.  The
// MFMA chain runs over k in ascending order of 32-wide steps.  The larger
// tiles re-read each operand from L2 fewer times (the forward of many samples).
template <int EPI, int KC, int BM, int BN>
__global__ void __launch_bounds__(256) k_gemm(const bf16* __restrict__ A, int lda, const bf16* __restrict__ Bt, int ldb,
                                              int ke, float* __restrict__ Cf, bf16* __restrict__ Cb, int ldc,
                                              const float* __restrict__ bias) {
    constexpr int PAD = 8;              // bf16 elements of row padding (LDS bank spread)
    constexpr int VR = KC / 8;          // 8-element vectors per tile row
    constexpr int NVA = BM * VR / 256;  // vectors per thread of the A tile
    constexpr int NVB = BN * VR / 256;  // and of the Bt tile
    constexpr int MT = BM / 32, NT = BN / 32;  // MFMA tiles per wave
    static_assert(KC % 32 == 0 && NVA >= 1 && NVB >= 1, "tile shape");
    __shared__ __align__(16) bf16 sA[BM][KC + PAD];
    __shared__ __align__(16) bf16 sB[BN][KC + PAD];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int wm = (BM / 2) * (w >> 1), wn = (BN / 2) * (w & 1);
    v4f acc[MT][NT];
    for (int i = 0; i < MT; ++i)
        for (int j = 0; j < NT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    // vector e = u*256 + t of a tile: row e / VR, k offset 8*(e % VR)
    v4u ra[NVA], rb[NVB];
    auto gload = [&](int k0) {
#pragma unroll
        for (int u = 0; u < NVA; ++u) {
            const int e = u * 256 + t, r = e / VR, kv = 8 * (e % VR);
            ra[u] = (k0 + kv < ke) ? *(const v4u*)&A[(size_t)(m0 + r) * lda + k0 + kv] : v4u{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int u = 0; u < NVB; ++u) {
            const int e = u * 256 + t, r = e / VR, kv = 8 * (e % VR);
            rb[u] = (k0 + kv < ke) ? *(const v4u*)&Bt[(size_t)(n0 + r) * ldb + k0 + kv] : v4u{0u, 0u, 0u, 0u};
        }
    };
    gload(0);
    for (int k0 = 0; k0 < ke; k0 += KC) {
        __syncthreads();  // the previous chunk's MFMAs have read LDS
#pragma unroll
        for (int u = 0; u < NVA; ++u) {
            const int e = u * 256 + t, r = e / VR, kv = 8 * (e % VR);
            *(v4u*)&sA[r][kv] = ra[u];
        }
#pragma unroll
        for (int u = 0; u < NVB; ++u) {
            const int e = u * 256 + t, r = e / VR, kv = 8 * (e % VR);
            *(v4u*)&sB[r][kv] = rb[u];
        }
        __syncthreads();
        if (k0 + KC < ke) gload(k0 + KC);
#pragma unroll
        for (int ks = 0; ks < KC; ks += 32) {
            v8bf a[MT], b[NT];
            for (int i = 0; i < MT; ++i) a[i] = *(const v8bf*)&sA[wm + 16 * i + (lane & 15)][ks + 8 * (lane >> 4)];
            for (int j = 0; j < NT; ++j) b[j] = *(const v8bf*)&sB[wn + 16 * j + (lane & 15)][ks + 8 * (lane >> 4)];
            for (int i = 0; i < MT; ++i)
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
    for (int i = 0; i < MT; ++i)
        for (int j = 0; j < NT; ++j)
            for (int r = 0; r < 4; ++r) {
                int row = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
                int col = n0 + wn + 16 * j + (lane & 15);
                size_t o = (size_t)row * ldc + col;
                float v = acc[i][j][r];
                if (EPI == EPI_BIAS_SILU) Cb[o] = f2bf(silu(v + bias[col]));
                else Cf[o] = v + bias[col];
            }
}

// The network's weights and biases as the one-kernel forward pass reads them.
struct MlpFwd {
    const bf16* wf[NLAYER];  // bf16 weights in MFMA operand order (frag_index)
    const float* b[NLAYER];
};

// Weights in operand order: lane l's 8 values of 16-column tile j and 32-wide
// k step s are one 16-byte vector, 64 lanes contiguous, so that an operand load
// is 1 KB of whole cache lines.  (From the transposed weights a load
// touched half of 16 lines, the other half needed a step later: a forward pass
// of 16 samples per workgroup took 17.1 us, 7.0 in this order.)  `steps`: k steps of the layer.
__host__ __device__ constexpr int frag_steps(int l) { return l == 0 ? 1 : NHID / 32; }
__host__ __device__ constexpr int frag_tiles(int l) { return l == NLAYER - 1 ? 1 : NHID / 16; }  // output: columns 0..15
__device__ __forceinline__ size_t frag_index(int tile, int step, int steps, int lane) {
    return ((size_t)(tile * steps + step) * 64 + lane) * 8;
}
// The backward products' order is that of W itself (a step covers 32 output
// columns; the output layer's first 32 of 64).
struct MlpFrag {
    const bf16* wb[NLAYER];
    bf16 *wf[NLAYER], *wb_frag[NLAYER];
};
__global__ void __launch_bounds__(256) k_frag(MlpFrag P) {
    int v = blockIdx.x * 256 + threadIdx.x;  // 16-byte vector over all layers
#pragma unroll
    for (int l = 0; l < NLAYER; ++l) {
        const int kin = l == 0 ? NIN_P : NHID, kout = l == NLAYER - 1 ? NOUT_P : NHID;
        const int steps = frag_steps(l), n = frag_tiles(l) * steps * 64;
        const int bsteps = l == NLAYER - 1 ? 1 : NHID / 32, nb = l == 0 ? 0 : NHID / 16 * bsteps * 64;
        const int lane = v & 63;
        if (v < n) {
            const int st = (v >> 6) % steps, tile = (v >> 6) / steps;
            const int k0 = 32 * st + 8 * (lane >> 4), col = 16 * tile + (lane & 15);
            for (int e = 0; e < 8; ++e) P.wf[l][(size_t)v * 8 + e] = k0 + e < kin ? P.wb[l][(size_t)(k0 + e) * kout + col] : 0;
            return;
        }
        v -= n;
        if (v < nb) {
            const int st = (v >> 6) % bsteps, tile = (v >> 6) / bsteps;
            for (int e = 0; e < 8; ++e)
                P.wb_frag[l][(size_t)v * 8 + e] = P.wb[l][(size_t)(16 * tile + (lane & 15)) * kout + 32 * st + 8 * (lane >> 4) + e];
            return;
        }
        v -= nb;
    }
}

// The whole forward pass of BM = 16 RT samples in one workgroup of NW waves,
// from the caller's fp32 inputs [n][9] to its fp32 outputs [n][5]: the
// activations of every hidden layer stay in LDS (BM x 256 bf16), so HBM sees
// the inputs, the outputs and (through L2) the weights.  Wave w computes columns
// 16 CT w .. of every layer for all rows, as RT x CT tiles of
// v_mfma_f32_16x16x32_bf16 with the weights as the first operand: lane l
// supplies 8 k's of output column l % 16 and of row l % 16, and receives the
// four consecutive columns 4 (l / 16) .. + 3 of row l % 16, so an epilogue
// packs four activations into one 8-byte LDS write.  The weights are loaded
// PF k steps ahead, across layer ends (they do not depend on the
// activations), the activations one step ahead, into register rings indexed by
// compile-time step numbers.  TWO: two activation buffers, one barrier per layer
// instead of two.
// Every product, sum order and epilogue is k_gemm's (the MFMA chain over k in
// ascending 32-wide steps from zero, the 16-wide input layer through one MFMA
// with k 16..31 zero), so the outputs are those of the layer-by-layer pass
// bit for bit.  LDS rows are 512 bytes with no padding; the 16-byte vector v
// of row r is stored at v ^ (r & 15), so the 16 rows an MFMA operand load
// reads fall in different banks.  Rows past n read zero inputs and are not
// stored.
// Shapes and what bounds them: see forward_fused.
__device__ __forceinline__ int swz(int r, int k) { return (((k >> 3) ^ (r & 15)) << 3) | (k & 7); }

template <int RT, int NW, int PF, bool TWO>
__global__ void __launch_bounds__(64 * NW) k_mlp_forward(const float* __restrict__ x, int n, MlpFwd P,
                                                         float* __restrict__ y) {
    constexpr int BM = 16 * RT, CT = 16 / NW;
    constexpr int NSTEP = NHID / 32, NHL = NLAYER - 2;  // k steps per layer, hidden 256 -> 256 layers
    __shared__ __align__(16) bf16 sH[TWO ? 2 : 1][BM][NHID];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int m0 = blockIdx.x * BM, c0 = 16 * CT * w;
    const int lr = lane & 15, q = lane >> 4, lk = 8 * q;
    v4f acc[RT][CT];
    v4f bias[CT];
    auto load_bias = [&](int l) {
#pragma unroll
        for (int j = 0; j < CT; ++j) bias[j] = *(const v4f*)&P.b[l][c0 + 16 * j + 4 * q];
    };
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    };
    // bias + SiLU of this wave's tile into the activation rows
    auto store_silu = [&](bf16(*h)[NHID]) {
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const int row = 16 * i + lr, col = c0 + 16 * j + 4 * q;
                const v4f v = acc[i][j] + bias[j];
                const v4f s = {silu(v.x), silu(v.y), silu(v.z), silu(v.w)};
                *(v4bf*)&h[row][swz(row, col)] = __builtin_convertvector(s, v4bf);
            }
    };
    v8bf B[PF + 1][CT], Am[2][RT];
    auto load_b = [&](int g) {  // weights of flat step g (layer 1 + g / NSTEP)
        const bf16* wf = P.wf[1 + g / NSTEP];
#pragma unroll
        for (int j = 0; j < CT; ++j) B[g % (PF + 1)][j] = *(const v8bf*)&wf[frag_index(CT * w + j, g % NSTEP, NSTEP, lane)];
    };
    // layer 0: k = 16 packed inputs (9 used), k 16..31 of the MFMA zero
    {
        v8bf b[CT], a[RT];
#pragma unroll
        for (int j = 0; j < CT; ++j)
            b[j] = *(const v8bf*)&P.wf[0][frag_index(CT * w + j, 0, 1, lane)];
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const int row = m0 + 16 * i + lr;
            v8f f = {};
            if (row < n && q < 2) {
                const float* xr = x + (size_t)row * NIN + lk;
#pragma unroll
                for (int k = 0; k < 8; ++k) f[k] = (k == 0 || q == 0) ? xr[k * (q == 0)] : 0.f;
            }
            a[i] = __builtin_convertvector(f, v8bf);
        }
        load_bias(0);
#pragma unroll
        for (int g = 0; g < PF; ++g) load_b(g);
        clear();
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
    }
    store_silu(sH[0]);
    __syncthreads();
#pragma unroll
    for (int h = 0; h < NHL; ++h) {
        bf16(*src)[NHID] = sH[TWO ? h & 1 : 0];
        auto load_a = [&](int ks, v8bf* dst) {
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const int row = 16 * i + lr;
                dst[i] = *(const v8bf*)&src[row][swz(row, ks + lk)];
            }
        };
        load_bias(1 + h);
        clear();
        load_a(0, Am[0]);
#pragma unroll
        for (int st = 0; st < NSTEP; ++st) {
            const int g = h * NSTEP + st;
            if (g + PF < NHL * NSTEP) load_b(g + PF);
            if (st + 1 < NSTEP) load_a(32 * (st + 1), Am[(st + 1) & 1]);
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(B[g % (PF + 1)][j], Am[st & 1][i], acc[i][j], 0, 0, 0);
        }
        if (!TWO) __syncthreads();  // every wave has read this layer's input
        store_silu(sH[TWO ? (h + 1) & 1 : 0]);
        __syncthreads();
    }
    // output layer: the first 16 of the padded 64 columns, row tiles dealt to the waves
    const bf16(*src)[NHID] = sH[TWO ? NHL & 1 : 0];
    const v4f bo = *(const v4f*)&P.b[NLAYER - 1][4 * q];
    for (int i = w; i < RT; i += NW) {
        v4f o = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NHID; ks += 32) {
            const v8bf b = *(const v8bf*)&P.wf[NLAYER - 1][frag_index(0, ks / 32, NSTEP, lane)];
            const v8bf a = *(const v8bf*)&src[16 * i + lr][swz(16 * i + lr, ks + lk)];
            o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, o, 0, 0, 0);
        }
        o += bo;
        const int row = m0 + 16 * i + lr;
        if (row < n) {
            float* yr = y + (size_t)row * NOUT;
            if (q == 0) { yr[0] = o.x; yr[1] = o.y; yr[2] = o.z; yr[3] = o.w; }
            if (q == 1) yr[4] = o.x;
        }
    }
}

// out[c][r] = in[r][c] for an R x Cc bf16 matrix; rows R..Rp-1 of the output's
// transposed shape (columns of `in` beyond Cc) are zero-filled up to Cp.
__global__ void k_transpose(const bf16* in, int R, int Cc, bf16* out, int Cp) {
    __shared__ bf16 tile[32][33];
    int bx = blockIdx.x * 32, by = blockIdx.y * 32;
    for (int k = threadIdx.y; k < 32; k += 8) {
        int r = by + k, c = bx + threadIdx.x;
        tile[k][threadIdx.x] = (r < R && c < Cc) ? in[(size_t)r * Cc + c] : (bf16)0;
    }
    __syncthreads();
    for (int k = threadIdx.y; k < 32; k += 8) {
        int c = bx + k, r = by + threadIdx.x;
        if (c < Cp && r < R) out[(size_t)c * R + r] = tile[threadIdx.x][k];
    }
}

__global__ void k_copy_floats(const float* a, int n, float* b) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = a[i];
}

// Inputs fp32 [n][NIN] -> bf16 [Mp][NIN_P] (zero padded).
__global__ void k_pack_inputs(const float* x, int n, int Mp, bf16* out) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= Mp * NIN_P) return;
    int r = i / NIN_P, c = i % NIN_P;
    out[i] = (r < n && c < NIN) ? f2bf(x[(size_t)r * NIN + c]) : (bf16)0;
}

// ---- training: three kernels per step (gradients, weight products, update)

// Layer l's increment in the parameter vector's layout (W[kin][kout], b[kout], ...).
__host__ __device__ constexpr int lay_kin(int l) { return l == 0 ? NIN_P : NHID; }
__host__ __device__ constexpr int lay_kout(int l) { return l == NLAYER - 1 ? NOUT_P : NHID; }
__host__ __device__ constexpr int lay_off(int l) {
    int o = 0;
    for (int k = 0; k < l; ++k) o += lay_kin(k) * lay_kout(k) + lay_kout(k);
    return o;
}
// Columns of a layer's pre-activation gradient that are kept (the output
// layer's padding columns are zero beyond the first 16).
__host__ __device__ constexpr int lay_gcols(int l) { return l == NLAYER - 1 ? 16 : NHID; }

struct MlpTrain {
    const bf16 *wf[NLAYER], *wb_frag[NLAYER];  // weights in operand order, forward and backward products
    const float* b[NLAYER];
    bf16 *hT[NLAYER], *gT[NLAYER];  // layer inputs and pre-activation gradients, [feature][sample]
    float* cs[NLAYER];              // column sums of the fp32 gradients over 16 samples: [Mp / 16][lay_gcols]
    float* lpart;                   // squared errors of 4 samples each
    const float *x, *t;             // samples [..][9], targets [..][5]
    const int* idx;                 // sample of each row (null: the row)
    int n, Mp;                      // samples, and rounded up to 64 (the rest zero rows without loss)
};

// Forward and backward of BM = 16 RT samples in one workgroup: the forward pass
// as k_mlp_forward, the pre-activations staying in registers (a lane holds the
// same tile of every layer, so SiLU' of the backward pass finds them in place),
// then from the output error down g_{l-1} = (g_l W_l^T) silu'(z_{l-1}), the
// gradients through LDS like the activations.  HBM sees the samples, the weights
// (L2), and what the weight products need: both factors transposed (sample
// contiguous), in 32-byte pieces written from LDS.
// Bound by the chain of 11 products in a workgroup, each step of which waits for
// its weights from L2 and for the LDS exchange between layers.  Shapes measured
// (us per training step, all three kernels, at 64 / 1024 / 4096 / 8192 samples):
// <1,8,8> 32 / 42 / 49 / 78, <2,8,3> 39 / 50 / 54 / 68, <2,8,8> (weights further
// ahead, but 50 registers spilled) 44 / 53 / 62 / 77, <2,16,4> 43 / 52 / 59 / 73,
// <1,4,4> 37 / 48 / 57 / 95.  So 16 samples a workgroup while those are no more
// than the 256 CUs, and 32 beyond.  A step of separate kernels for every product,
// transpose, column sum and update (75 launches) took 404 us at 8192 samples.
// The arithmetic is that of separate products: MFMA chains over k in ascending
// 32-wide steps, fp32 epilogues, column sums of 16 samples in order.
template <int RT, int NW, int PF>
__global__ void __launch_bounds__(64 * NW) k_mlp_grad(MlpTrain P) {
    constexpr int BM = 16 * RT, CT = 16 / NW;
    constexpr int NSTEP = NHID / 32, NHL = NLAYER - 2, NF = NHL * NSTEP;  // forward steps 0..NF-1, backward NF..2NF-1
    constexpr int GP = NHID + 4;  // fp32 gradient row, padded
    static_assert(NW * 64 >= NHID * RT, "a thread per column and 16 samples");
    __shared__ __align__(16) bf16 sH[2][BM][NHID];
    __shared__ __align__(16) float sG[2][BM][GP];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int m0 = blockIdx.x * BM, c0 = 16 * CT * w;
    const int lr = lane & 15, q = lane >> 4, lk = 8 * q;
    v4f z[NLAYER - 1][RT][CT];
    v8bf B[PF + 1][CT], Am[2][RT];
    auto load_b = [&](int g) {  // weights of flat step g
        const bf16* wf = g < NF ? P.wf[1 + g / NSTEP] : P.wb_frag[NHL - (g - NF) / NSTEP];
#pragma unroll
        for (int j = 0; j < CT; ++j) B[g % (PF + 1)][j] = *(const v8bf*)&wf[frag_index(CT * w + j, g % NSTEP, NSTEP, lane)];
    };
    // eight k steps against the activations (or gradients) in src, from flat step g0
    auto product = [&](v4f(*acc)[CT], bf16(*src)[NHID], int g0) {
        auto load_a = [&](int ks, v8bf* dst) {
#pragma unroll
            for (int i = 0; i < RT; ++i) dst[i] = *(const v8bf*)&src[16 * i + lr][swz(16 * i + lr, ks + lk)];
        };
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        load_a(0, Am[0]);
#pragma unroll
        for (int st = 0; st < NSTEP; ++st) {
            const int g = g0 + st;
            if (g + PF < 2 * NF) load_b(g + PF);
            if (st + 1 < NSTEP) load_a(32 * (st + 1), Am[(st + 1) & 1]);
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(B[g % (PF + 1)][j], Am[st & 1][i], acc[i][j], 0, 0, 0);
        }
    };
    // column t % 256, samples 16 (t / 256) .. + 15 of an LDS tile, to [feature][sample]
    const int tg = t / NHID, tc = NW * 64 == NHID * RT || tg < RT ? t & (NHID - 1) : NHID;
    auto put16 = [&](bf16* dst, const v8bf& a, const v8bf& b) {
        v8bf* o = reinterpret_cast<v8bf*>(dst + m0 + 16 * tg);
        o[0] = a;
        o[1] = b;
    };
    auto store_hT = [&](bf16(*h)[NHID], bf16* dst) {
        if (tc >= NHID) return;
        v8us a, b;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            a[k] = h[16 * tg + k][swz(16 * tg + k, tc)];
            b[k] = h[16 * tg + 8 + k][swz(16 * tg + 8 + k, tc)];
        }
        put16(dst + (size_t)tc * P.Mp, __builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b));
    };
    auto store_gT = [&](float(*g)[GP], int l, int cols) {
        if (tc >= cols) return;
        v8f a, b;
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) { a[k] = g[16 * tg + k][tc]; s += a[k]; }
#pragma unroll
        for (int k = 0; k < 8; ++k) { b[k] = g[16 * tg + 8 + k][tc]; s += b[k]; }
        P.cs[l][(size_t)(m0 / 16 + tg) * cols + tc] = s;
        put16(P.gT[l] + (size_t)tc * P.Mp, __builtin_convertvector(a, v8bf), __builtin_convertvector(b, v8bf));
    };
    // ---- forward.  Layer 0: k = 16 packed inputs (9 used), k 16..31 of the MFMA zero
    {
        v8bf a[RT];
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const int row = m0 + 16 * i + lr;
            v8f f = {};
            if (row < P.n && q < 2) {
                const float* xr = P.x + (size_t)(P.idx ? P.idx[row] : row) * NIN + lk;
#pragma unroll
                for (int k = 0; k < 8; ++k) f[k] = (k == 0 || q == 0) ? xr[k * (q == 0)] : 0.f;
            }
            a[i] = __builtin_convertvector(f, v8bf);
            if (w == 0 && q < 2) *(v8bf*)&sH[1][16 * i + lr][swz(16 * i + lr, lk)] = a[i];
        }
#pragma unroll
        for (int g = 0; g < PF; ++g) load_b(g);
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            const v8bf b = *(const v8bf*)&P.wf[0][frag_index(CT * w + j, 0, 1, lane)];
#pragma unroll
            for (int i = 0; i < RT; ++i)
                z[0][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a[i], v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        }
    }
#pragma unroll
    for (int l = 0; l < NLAYER - 1; ++l) {
        if (l > 0) product(z[l], sH[(l - 1) & 1], (l - 1) * NSTEP);
        // (layer 0's packed inputs lie in buffer 1 until layer 1 has been computed)
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            const v4f bias = *(const v4f*)&P.b[l][c0 + 16 * j + 4 * q];
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const int row = 16 * i + lr, col = c0 + 16 * j + 4 * q;
                const v4f v = z[l][i][j] + bias;
                z[l][i][j] = v;
                const v4f h = {silu(v.x), silu(v.y), silu(v.z), silu(v.w)};
                *(v4bf*)&sH[l & 1][row][swz(row, col)] = __builtin_convertvector(h, v4bf);
            }
        }
        __syncthreads();
        if (l == 0 && tc < NIN_P) store_hT(sH[1], P.hT[0]);
        store_hT(sH[l & 1], P.hT[l + 1]);
        if (l == 0) __syncthreads();  // the inputs are out before layer 1 overwrites them
    }
    // output layer (first 16 columns), error and loss: wave i takes row tile i
    constexpr int LB = (NLAYER - 2) & 1;  // buffer of the last activations
    if (w < RT) {
        const int i = w, row = m0 + 16 * i + lr;
        v4f o = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NHID; ks += 32) {
            const v8bf b = *(const v8bf*)&P.wf[NLAYER - 1][frag_index(0, ks / 32, NSTEP, lane)];
            const v8bf a = *(const v8bf*)&sH[LB][16 * i + lr][swz(16 * i + lr, ks + lk)];
            o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, o, 0, 0, 0);
        }
        o += *(const v4f*)&P.b[NLAYER - 1][4 * q];
        v4f g = {}, e2 = {};
        if (row < P.n) {
            const float* tr = P.t + (size_t)(P.idx ? P.idx[row] : row) * NOUT;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (4 * q + c < NOUT) {
                    const float d = o[c] - tr[4 * q + c];
                    e2[c] = d * d;
                    g[c] = 2.0f * d / (float)(P.n * NOUT);
                }
        }
        // loss of rows 4k .. 4k + 3: per column (0 + 2) + (1 + 3), then ((c0 + c4) + c2) + (c1 + c3)
        v4f r;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float u = e2[c] + __shfl_xor(e2[c], 2);
            r[c] = u + __shfl_xor(u, 1);
        }
        const float r4 = __shfl(r.x, (lane & 15) + 16);  // column 4
        if (q == 0 && (lr & 3) == 0) P.lpart[row / 4] = ((r.x + r4) + r.z) + (r.y + r.w);
        *(v4f*)&sG[0][16 * i + lr][4 * q] = g;
        *(v4bf*)&sH[1 - LB][16 * i + lr][swz(16 * i + lr, 4 * q)] = __builtin_convertvector(g, v4bf);
        *(v4bf*)&sH[1 - LB][16 * i + lr][swz(16 * i + lr, 16 + 4 * q)] = v4bf{};  // k 16..31 of the one step below
    }
    __syncthreads();
    // ---- backward: g of layer l - 1 from that of layer l
    store_gT(sG[0], NLAYER - 1, 16);
#pragma unroll
    for (int l = NLAYER - 1; l >= 1; --l) {
        const int src = (NLAYER - 1 - l + 1 - LB) & 1, dst = 1 - src, gb = (NLAYER - l) & 1;
        v4f acc[RT][CT];
        if (l == NLAYER - 1) {  // 16 of the 64 padded columns are not zero: one step
#pragma unroll
            for (int j = 0; j < CT; ++j) {
                const v8bf b = *(const v8bf*)&P.wb_frag[l][frag_index(CT * w + j, 0, 1, lane)];
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const v8bf a = *(const v8bf*)&sH[src][16 * i + lr][swz(16 * i + lr, lk)];
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                }
            }
        } else {
            product(acc, sH[src], NF + (NHL - l) * NSTEP);
        }
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const int row = 16 * i + lr, col = c0 + 16 * j + 4 * q;
                const v4f v = acc[i][j], zz = z[l - 1][i][j];
                const v4f g = {v.x * dsilu(zz.x), v.y * dsilu(zz.y), v.z * dsilu(zz.z), v.w * dsilu(zz.w)};
                *(v4f*)&sG[gb][row][col] = g;
                if (l > 1) *(v4bf*)&sH[dst][row][swz(row, col)] = __builtin_convertvector(g, v4bf);
            }
        __syncthreads();
        store_gT(sG[gb], l - 1, NHID);
    }
}

// Weight gradients dW_l = H_l^T G_l of layers [l0, l1), split over the samples:
// one workgroup per 64 x 64 tile and split (blockIdx.y), all layers in one
// launch so that their tiles fill the GPU together (72 tiles x 8 splits at 8192
// samples: 19 us).  Bound by the operands from HBM/L2 (42 MB written just before).  Both factors lie with the sample contiguous; a chunk of 64 samples
// goes through LDS, the next one's loads under way.  The MFMA chain runs over
// the split's samples in ascending 32-wide steps.  part: layer l's
// [nsplit][lay_kin][lay_gcols] at its offset.
struct MlpWgrad {
    const bf16 *hT[NLAYER], *gT[NLAYER];
    float* part[NLAYER];
    int Mp, ks;  // samples, and per split (a multiple of 16)
};
__host__ __device__ constexpr int wg_tm(int l) { return l == 0 ? 1 : NHID / 64; }
__host__ __device__ constexpr int wg_tn(int l) { return l == NLAYER - 1 ? 1 : NHID / 64; }
__global__ void __launch_bounds__(256) k_wgrad(MlpWgrad P, int l0, int l1) {
    constexpr int KC = 64, PAD = 8, VR = KC / 8;
    __shared__ __align__(16) bf16 sA[64][KC + PAD];
    __shared__ __align__(16) bf16 sB[64][KC + PAD];
    int l = l0, tile = blockIdx.x;
    while (l + 1 < l1 && tile >= wg_tm(l) * wg_tn(l)) { tile -= wg_tm(l) * wg_tn(l); ++l; }
    const int m0 = 64 * (tile / wg_tn(l)), n0 = 64 * (tile % wg_tn(l));
    const int rows = lay_kin(l), cols = lay_gcols(l);
    const bf16 *A = P.hT[l], *Bt = P.gT[l];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int wm = 32 * (w >> 1), wn = 32 * (w & 1);
    const int kb = blockIdx.y * P.ks, ke = kb + P.ks;
    v4f acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    v4u ra[2], rb[2];
    auto gload = [&](int k0) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = u * 256 + t, r = e / VR, kv = k0 + 8 * (e % VR);
            ra[u] = kv < ke && m0 + r < rows ? *(const v4u*)&A[(size_t)(m0 + r) * P.Mp + kv] : v4u{0u, 0u, 0u, 0u};
            rb[u] = kv < ke && n0 + r < cols ? *(const v4u*)&Bt[(size_t)(n0 + r) * P.Mp + kv] : v4u{0u, 0u, 0u, 0u};
        }
    };
    gload(kb);
    for (int k0 = kb; k0 < ke; k0 += KC) {
        __syncthreads();  // the previous chunk's MFMAs have read LDS
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = u * 256 + t, r = e / VR, kv = 8 * (e % VR);
            *(v4u*)&sA[r][kv] = ra[u];
            *(v4u*)&sB[r][kv] = rb[u];
        }
        __syncthreads();
        if (k0 + KC < ke) gload(k0 + KC);
#pragma unroll
        for (int ks = 0; ks < KC; ks += 32) {
            v8bf a[2], b[2];
            for (int i = 0; i < 2; ++i) a[i] = *(const v8bf*)&sA[wm + 16 * i + (lane & 15)][ks + 8 * (lane >> 4)];
            for (int j = 0; j < 2; ++j) b[j] = *(const v8bf*)&sB[wn + 16 * j + (lane & 15)][ks + 8 * (lane >> 4)];
            for (int i = 0; i < 2; ++i)
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
    float* out = P.part[l] + (size_t)blockIdx.y * rows * cols;
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + wm + 16 * i + 4 * (lane >> 4) + r, col = n0 + wn + 16 * j + (lane & 15);
                if (row < rows && col < cols) out[(size_t)row * cols + col] = acc[i][j][r];
            }
}

// The end of a step for layers [l0, l1): the splits' partials added in order,
// then Adam on the fp32 weights with the bf16 copies refreshed (ADAM), or the
// gradient vector written.  A thread owns 8 columns of a weight row; further
// blocks own 64 bias columns each (the 16-sample sums of a 64-sample chunk in
// order, four lanes of every fourth chunk, then those in order) and the last one
// the loss (l0 = 0 only).  Bound by the partials (8.7 MB) and the optimiser state
// (10 MB with the bf16 copies) at 8192 samples: 14 us.
struct MlpUpdate {
    float *w[NLAYER], *m[NLAYER], *v[NLAYER], *b[NLAYER], *mb[NLAYER], *vb[NLAYER];
    bf16 *wb[NLAYER], *wf[NLAYER], *wb_frag[NLAYER];
    const float *part[NLAYER], *cs[NLAYER];
    const float* lpart;
    float *grad, *loss;
    int nsplit, Mp, n;
    float lr, b1, b2, eps, c1, c2;
};
__device__ __forceinline__ float adam(float w, float g, float* m, float* v, const MlpUpdate& P) {
    const float mi = P.b1 * *m + (1.f - P.b1) * g;
    const float vi = P.b2 * *v + (1.f - P.b2) * g * g;
    *m = mi;
    *v = vi;
    return w - P.lr * (mi * P.c1) / (sqrtf(vi * P.c2) + P.eps);
}
__host__ __device__ constexpr int upd_wblocks(int l) { return lay_kin(l) * lay_gcols(l) / 8 / 256 + (lay_kin(l) * lay_gcols(l) / 8 % 256 != 0); }
__host__ __device__ constexpr int upd_bblocks(int l) { return (lay_gcols(l) + 63) / 64; }
template <bool ADAM>
__global__ void __launch_bounds__(256) k_update(MlpUpdate P, int l0, int l1) {
    __shared__ double sm[256];
    int blk = blockIdx.x;
    const int t = threadIdx.x;
    for (int l = l0; l < l1; ++l) {
        const int cols = lay_gcols(l), kout = lay_kout(l);
        if (blk < upd_wblocks(l)) {
            const int e = blk * 256 + t, nv = lay_kin(l) * cols / 8;
            if (e >= nv) return;
            const int k = e / (cols / 8), c = 8 * (e % (cols / 8));
            const size_t n = (size_t)lay_kin(l) * cols, o = (size_t)k * cols + c, wo = (size_t)k * kout + c;
            v8f g = {};
            for (int s = 0; s < P.nsplit; ++s) g += *(const v8f*)&P.part[l][(size_t)s * n + o];
            if (!ADAM) {
                for (int u = 0; u < 8; ++u) P.grad[lay_off(l) + wo + u] = g[u];
                return;
            }
            v8f w = *(const v8f*)&P.w[l][wo], m = *(const v8f*)&P.m[l][wo], v = *(const v8f*)&P.v[l][wo];
            for (int u = 0; u < 8; ++u) {
                float mu = m[u], vu = v[u];
                w[u] = adam(w[u], g[u], &mu, &vu, P);
                m[u] = mu;
                v[u] = vu;
            }
            *(v8f*)&P.w[l][wo] = w;
            *(v8f*)&P.m[l][wo] = m;
            *(v8f*)&P.v[l][wo] = v;
            const v8bf h = __builtin_convertvector(w, v8bf);
            *(v8bf*)&P.wb[l][wo] = h;
            if (l > 0)  // backward operand: row k of tile k / 16, columns c .. c + 7 of step c / 32
                *(v8bf*)&P.wb_frag[l][frag_index(k / 16, c / 32, l == NLAYER - 1 ? 1 : NHID / 32, k % 16 + 16 * (c % 32 / 8))] = h;
            for (int u = 0; u < 8; ++u)  // forward operand: column c + u, k within step k / 32
                *(__bf16*)&P.wf[l][frag_index((c + u) / 16, k / 32, frag_steps(l), (c + u) % 16 + 16 * (k % 32 / 8)) + k % 8] = h[u];
            return;
        }
        blk -= upd_wblocks(l);
        if (blk < upd_bblocks(l)) {
            const int c = blk * 64 + (t & 63), r = t >> 6, chunks = P.Mp / 64;
            float s = 0.f;
            if (c < cols)
                for (int k = r; k < chunks; k += 4) {
                    const float* p = P.cs[l] + (size_t)4 * k * cols + c;
                    s += ((p[0] + p[cols]) + p[2 * (size_t)cols]) + p[3 * (size_t)cols];
                }
            float* sf = reinterpret_cast<float*>(sm);
            sf[t] = s;
            __syncthreads();
            if (r == 0 && c < cols) {
                const float g = ((sf[t] + sf[64 + t]) + sf[128 + t]) + sf[192 + t];
                if (ADAM) P.b[l][c] = adam(P.b[l][c], g, &P.mb[l][c], &P.vb[l][c], P);
                else P.grad[lay_off(l) + lay_kin(l) * kout + c] = g;
            }
            return;
        }
        blk -= upd_bblocks(l);
    }
    double s = 0.0;
    for (int i = t; i < P.Mp / 4; i += 256) s += P.lpart[i];
    sm[t] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (t < k) sm[t] += sm[t + k];
        __syncthreads();
    }
    if (t == 0) *P.loss = (float)(sm[0] * (1.0f / (float)(P.n * NOUT)));
}

// y[i][0..NOUT) of the padded output rows, packed densely for one host copy
__global__ void k_pack_outputs(const float* __restrict__ yp, int nsamp, float* __restrict__ y) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (size_t)nsamp * NOUT) y[i] = yp[(i / NOUT) * NOUT_P + i % NOUT];
}

__global__ void k_to_bf16(const float* a, size_t n, bf16* b) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = f2bf(a[i]);
}

}  // namespace ofx

using namespace ofx;

struct ofx_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    int kin[NLAYER], kout[NLAYER];        // padded shapes of each layer
    float *w[NLAYER], *b[NLAYER];          // fp32 master
    bf16 *wb[NLAYER], *wt[NLAYER];         // bf16 copy and its transpose
    bf16 *wf[NLAYER], *wb_frag[NLAYER];    // bf16 copies in MFMA operand order (frag_index)
    float *mw[NLAYER], *vw[NLAYER], *mb[NLAYER], *vb[NLAYER];
    float* grad = nullptr;                 // gradient vector, in the parameters' layout
    int step = 0;
    // layered forward pass, sized for `cap` samples
    int cap = 0;
    bf16* h[NLAYER];                       // layer inputs: h[0] = packed inputs
    float *y = nullptr, *yd = nullptr;     // padded and dense outputs
    float* xin = nullptr;
    std::vector<void*> fwd_allocs;
    // gradients, sized for `tcap` samples: one block (MlpTrain, MlpWgrad)
    int tcap = 0;
    char* tbuf = nullptr;
    bf16 *hT[NLAYER], *gT[NLAYER];
    float *cs[NLAYER], *lpart = nullptr, *part = nullptr, *loss = nullptr, *tx = nullptr, *tt = nullptr;
    float *io_x = nullptr, *io_y = nullptr;  // device copies of a one-kernel forward's inputs and outputs
    int io_cap = 0;
    hipStream_t out_stream = nullptr;        // outputs of a piped forward pass
    hipEvent_t out_ready[8] = {};            // a piece's outputs are computed
    int fwd_variant = 1;  // inference forward pass: 0 layer by layer, 1 one kernel (k_mlp_forward)
    std::vector<void*> allocs;
};

namespace {

int mlp_alloc(ofx_mlp* n, void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) { set_error("mlp: out of device memory"); return OFX_ENOMEM; }
    n->allocs.push_back(*p);
    OFX_HIP(hipMemsetAsync(*p, 0, bytes, n->stream));
    return 0;
}

// Buffers of a layered forward pass.
int layered_reserve(ofx_mlp* n, int samples) {
    const int Mp = (samples + 63) / 64 * 64;
    if (Mp <= n->cap) return 0;
    OFX_HIP(hipStreamSynchronize(n->stream));
    for (void* p : n->fwd_allocs) (void)hipFree(p);
    n->fwd_allocs.clear();
    n->cap = 0;
    auto A = [&](void** p, size_t bytes) -> int {
        if (hipMalloc(p, bytes) != hipSuccess) { set_error("mlp: out of device memory"); return OFX_ENOMEM; }
        n->fwd_allocs.push_back(*p);
        return 0;
    };
    for (int l = 0; l < NLAYER; ++l) OFX_TRY(A((void**)&n->h[l], sizeof(bf16) * (size_t)Mp * n->kin[l]));
    OFX_TRY(A((void**)&n->y, sizeof(float) * (size_t)Mp * NOUT_P));
    OFX_TRY(A((void**)&n->yd, sizeof(float) * (size_t)Mp * NOUT));
    OFX_TRY(A((void**)&n->xin, sizeof(float) * (size_t)Mp * NIN));
    n->cap = Mp;
    return 0;
}

// Splits of a weight gradient over Mp samples: at most SPLITK_CHUNK samples each
// while Mp divides into multiples of 16.
int wgrad_splits(int Mp) {
    int ns = 1;
    while (Mp / ns > SPLITK_CHUNK && Mp % (ns * 2) == 0 && (Mp / (ns * 2)) % 16 == 0) ns *= 2;
    return ns;
}
// All layers' partials together up to this many splits, one layer's beyond
// (64: 70 MB; 128 more layers' tiles in flight would not fill the GPU any better).
constexpr int SPLITS_TOGETHER = 64;
constexpr int wgrad_elems(int l) { return lay_kin(l) * lay_gcols(l); }

// Buffers of the gradients of `samples` samples (every element a kernel reads is
// written first).
int train_reserve(ofx_mlp* n, int samples) {
    const int Mp = (samples + 63) / 64 * 64;
    if (Mp <= n->tcap) return 0;
    OFX_HIP(hipStreamSynchronize(n->stream));
    if (n->tbuf) (void)hipFree(n->tbuf);
    n->tbuf = nullptr;
    n->tcap = 0;
    // a smaller call may split into more pieces than a larger one (an odd
    // multiple of 64 stops early), so the partials are sized for any size up to Mp:
    // wgrad_splits(m) < 2 m / SPLITK_CHUNK + 1
    const size_t ns = 2 * (size_t)(Mp / SPLITK_CHUNK) + 1;
    size_t all = 0, one = 0;
    for (int l = 0; l < NLAYER; ++l) { all += wgrad_elems(l); one = std::max<size_t>(one, wgrad_elems(l)); }
    const size_t pel = std::max(std::min<size_t>(ns, SPLITS_TOGETHER) * all, ns * one);
    size_t o = 0;
    auto take = [&](size_t bytes) { size_t at = o; o += (bytes + 255) / 256 * 256; return at; };
    size_t hT[NLAYER], gT[NLAYER], cs[NLAYER];
    for (int l = 0; l < NLAYER; ++l) {
        hT[l] = take(sizeof(bf16) * (size_t)Mp * lay_kin(l));
        gT[l] = take(sizeof(bf16) * (size_t)Mp * lay_gcols(l));
        cs[l] = take(sizeof(float) * (size_t)(Mp / 16) * lay_gcols(l));
    }
    const size_t lp = take(sizeof(float) * (size_t)(Mp / 4)), lo = take(sizeof(float)), pa = take(sizeof(float) * pel),
                 tx = take(sizeof(float) * (size_t)Mp * NIN), tt = take(sizeof(float) * (size_t)Mp * NOUT);
    if (hipMalloc((void**)&n->tbuf, o) != hipSuccess) {
        n->tbuf = nullptr;
        set_error("mlp: out of device memory");
        return OFX_ENOMEM;
    }
    for (int l = 0; l < NLAYER; ++l) {
        n->hT[l] = (bf16*)(n->tbuf + hT[l]);
        n->gT[l] = (bf16*)(n->tbuf + gT[l]);
        n->cs[l] = (float*)(n->tbuf + cs[l]);
    }
    n->lpart = (float*)(n->tbuf + lp);
    n->loss = (float*)(n->tbuf + lo);
    n->part = (float*)(n->tbuf + pa);
    n->tx = (float*)(n->tbuf + tx);
    n->tt = (float*)(n->tbuf + tt);
    n->tcap = Mp;
    return 0;
}

// Device buffers of a one-kernel forward of `samples` samples.
int io_reserve(ofx_mlp* n, int samples) {
    if (samples <= n->io_cap) return 0;
    OFX_HIP(hipStreamSynchronize(n->stream));
    if (n->io_x) (void)hipFree(n->io_x);
    n->io_x = nullptr;
    n->io_cap = 0;
    if (hipMalloc((void**)&n->io_x, sizeof(float) * (size_t)samples * (NIN + NOUT)) != hipSuccess) {
        n->io_x = nullptr;
        set_error("mlp: out of device memory");
        return OFX_ENOMEM;
    }
    n->io_y = n->io_x + (size_t)samples * NIN;
    n->io_cap = samples;
    return 0;
}

// C = A Bt^T (see k_gemm): A [M][K], Bt [N][K].
template <int EPI>
int gemm_on(hipStream_t st, const bf16* A, int lda, const bf16* Bt, int ldb, int M, int N, int K, float* Cf, bf16* Cb,
            int ldc, const float* bias) {
    if (M % 64 || N % 64 || K % 16) {
        set_error("mlp: GEMM shape not tiled");
        return OFX_EINVAL;
    }
    // 128-row tiles (and 128 columns where N allows) once there are rows
    // enough to fill the GPU with them: fewer L2 re-reads of both operands
    if (M % 128 == 0 && M >= 65536 && K % 64 == 0) {
        if (N % 128 == 0) k_gemm<EPI, 64, 128, 128><<<dim3(N / 128, M / 128), 256, 0, st>>>(A, lda, Bt, ldb, K, Cf, Cb, ldc, bias);
        else k_gemm<EPI, 64, 128, 64><<<dim3(N / 64, M / 128), 256, 0, st>>>(A, lda, Bt, ldb, K, Cf, Cb, ldc, bias);
    } else {
        dim3 grid(N / 64, M / 64);
        if (K % 64 == 0) k_gemm<EPI, 64, 64, 64><<<grid, 256, 0, st>>>(A, lda, Bt, ldb, K, Cf, Cb, ldc, bias);
        else k_gemm<EPI, 32, 64, 64><<<grid, 256, 0, st>>>(A, lda, Bt, ldb, K, Cf, Cb, ldc, bias);
    }
    OFX_HIP(hipGetLastError());
    return 0;
}

// All layers on packed inputs in [Mp][16] -> padded outputs yp [Mp][64]; layer
// l's output in act(l).
template <class ACT>
int forward_layered(const ofx_mlp* n, hipStream_t st, const bf16* in, int Mp, ACT act, float* yp) {
    const bf16* h = in;
    for (int l = 0; l < NLAYER - 1; ++l) {
        OFX_TRY(gemm_on<EPI_BIAS_SILU>(st, h, n->kin[l], n->wt[l], n->kin[l], Mp, n->kout[l], n->kin[l], nullptr, act(l),
                                       n->kout[l], n->b[l]));
        h = act(l);
    }
    const int L = NLAYER - 1;
    return gemm_on<EPI_BIAS>(st, h, n->kin[L], n->wt[L], n->kin[L], Mp, n->kout[L], n->kin[L], yp, nullptr, n->kout[L],
                             n->b[L]);
}

int transpose(ofx_mlp* n, const bf16* in, int R, int C, bf16* out, int Cp) {
    dim3 grid((std::max(C, Cp) + 31) / 32, (R + 31) / 32);
    k_transpose<<<grid, dim3(32, 8), 0, n->stream>>>(in, R, C, out, Cp);
    OFX_HIP(hipGetLastError());
    return 0;
}

// All layers in one kernel (k_mlp_forward): fp32 inputs x [n][9] -> fp32 outputs
// y [n][5].
template <int RT, int NW, int PF, bool TWO>
int forward_shape(const ofx_mlp* n, hipStream_t st, const float* x, int nsamp, float* y) {
    MlpFwd P;
    for (int l = 0; l < NLAYER; ++l) { P.wf[l] = n->wf[l]; P.b[l] = n->b[l]; }
    k_mlp_forward<RT, NW, PF, TWO><<<(nsamp + 16 * RT - 1) / (16 * RT), 64 * NW, 0, st>>>(x, nsamp, P, y);
    OFX_HIP(hipGetLastError());
    return 0;
}
// Rows per workgroup by sample count.  Up to one workgroup per CU the pass is
// bound by one workgroup's chain (five layers of weights through one CU, ~1 us
// each), shortest with the fewest rows; beyond, by the SiLU epilogues, the
// matrix units and the weights' L2 traffic, which more rows share.  us for 16 /
// 32 / 64 rows: 500 samples 7.2 / 9.2 / 12.9, 4096 8.3 / 9.6 / 13.2, 8192 13.5 /
// 10.2 / 13.5, 16384 24 / 17 / 15, 1,000,003 1186 / 803 / 627 (0.89 PFLOP/s).
// 128 rows: 710; four waves of 64 columns instead of eight of 32: 643.  With the
// weights' transposed rows as operands, activations packed and written one
// by one, and separate kernels packing inputs and outputs, 500 samples took
// 37 us and 1,000,003 took 1333.
int forward_fused(const ofx_mlp* n, hipStream_t st, const float* x, int nsamp, float* y) {
    if (nsamp <= 16 * 256) return forward_shape<1, 8, 8, true>(n, st, x, nsamp, y);
    if (nsamp <= 32 * 256) return forward_shape<2, 8, 8, true>(n, st, x, nsamp, y);
    return forward_shape<4, 8, 4, true>(n, st, x, nsamp, y);
}

// Whether inputs x and outputs y of n samples share memory: the one-kernel pass
// writes rows while it reads others, and the piped one while others are not uploaded.
bool overlapping(const float* x, const float* y, int n) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(x), b = reinterpret_cast<uintptr_t>(y);
    return a < b + sizeof(float) * (size_t)n * NOUT && b < a + sizeof(float) * (size_t)n * NIN;
}

// A forward pass of many host samples in pieces: this thread copies a piece's
// inputs and launches its kernel, a second one copies finished pieces' outputs.
// Copies of ordinary host memory hold the calling thread (1.2 ms in, 1.2 ms out,
// as much again for the first touch of a new output array, at 1,000,003
// samples, next to 0.63 ms of computing), so one after another they were most
// of a call.  us in one piece / piped: 140,000 samples 435 / 490, 300,000
// 880 / 790, 500,000 1400 / 1150, 1,000,003 3000 / 2000; pieces of 65,536 there 2130.
// Returns OFX_ESTATE, having done nothing, where no second thread or stream can be had.
constexpr int PIPE_PIECE = 1 << 17, PIPE_MIN = 1 << 18;
static_assert(MLP_MAXN <= 8 * PIPE_PIECE, "an event per piece");
int forward_piped(ofx_mlp* n, const float* x, int nsamp, float* y) {
    const int np = (nsamp + PIPE_PIECE - 1) / PIPE_PIECE;
    if (!n->out_stream && hipStreamCreateWithFlags(&n->out_stream, hipStreamNonBlocking) != hipSuccess) {
        n->out_stream = nullptr;
        (void)hipGetLastError();  // the caller goes on without
        return OFX_ESTATE;
    }
    for (int p = 0; p < np; ++p)
        if (!n->out_ready[p] && hipEventCreateWithFlags(&n->out_ready[p], hipEventDisableTiming) != hipSuccess) {
            n->out_ready[p] = nullptr;
            (void)hipGetLastError();
            return OFX_ESTATE;
        }
    std::mutex mu;
    std::condition_variable cv;
    int launched = 0;      // pieces whose event is recorded
    bool failed = false;   // no more will come
    hipError_t out = hipSuccess;
    auto count = [&](int p) { return std::min(PIPE_PIECE, nsamp - p * PIPE_PIECE); };
    auto outputs = [&]() {
        out = hipSetDevice(n->device);
        for (int p = 0; p < np && out == hipSuccess; ++p) {
            {
                std::unique_lock<std::mutex> lock(mu);
                cv.wait(lock, [&] { return launched > p || failed; });
                if (launched <= p) break;
            }
            const size_t o = (size_t)p * PIPE_PIECE * NOUT;
            out = hipStreamWaitEvent(n->out_stream, n->out_ready[p], 0);
            if (out == hipSuccess)
                out = hipMemcpyAsync(y + o, n->io_y + o, sizeof(float) * (size_t)count(p) * NOUT, hipMemcpyDeviceToHost,
                                     n->out_stream);
        }
        const hipError_t done = hipStreamSynchronize(n->out_stream);  // (also after an error: y is the caller's again)
        if (out == hipSuccess) out = done;
        (void)hipGetLastError();  // reported by the caller's thread
    };
    std::thread worker;
    try {
        worker = std::thread(outputs);
    } catch (...) {  // no thread, or no memory for one
        return OFX_ESTATE;
    }
    int rc = 0;
    for (int p = 0; p < np && !rc; ++p) {
        const size_t o = (size_t)p * PIPE_PIECE * NIN;
        if (hipMemcpyAsync(n->io_x + o, x + o, sizeof(float) * (size_t)count(p) * NIN, hipMemcpyHostToDevice, n->stream) !=
            hipSuccess)
            rc = OFX_EHIP;
        if (!rc) rc = forward_fused(n, n->stream, n->io_x + o, count(p), n->io_y + (size_t)p * PIPE_PIECE * NOUT);
        if (!rc && hipEventRecord(n->out_ready[p], n->stream) != hipSuccess) rc = OFX_EHIP;
        {
            std::lock_guard<std::mutex> lock(mu);
            if (rc) failed = true;
            else launched = p + 1;
        }
        cv.notify_one();
    }
    worker.join();
    if (hipStreamSynchronize(n->stream) != hipSuccess || out != hipSuccess) rc = OFX_EHIP;
    if (rc == OFX_EHIP) {
        (void)hipGetLastError();  // reported here
        set_error("mlp_forward: HIP error");
    }
    return rc;
}

// The operand-ordered weights of the one-kernel forward and of training.
int refresh_frag(ofx_mlp* n) {
    MlpFrag P;
    int vec = 0;
    for (int l = 0; l < NLAYER; ++l) {
        P.wb[l] = n->wb[l]; P.wf[l] = n->wf[l]; P.wb_frag[l] = n->wb_frag[l];
        vec += 64 * frag_tiles(l) * frag_steps(l) + (l == 0 ? 0 : 64 * (NHID / 16) * (l == NLAYER - 1 ? 1 : NHID / 32));
    }
    k_frag<<<(vec + 255) / 256, 256, 0, n->stream>>>(P);
    OFX_HIP(hipGetLastError());
    return 0;
}

// The transposed bf16 weights [kout][kin] that the layered forward products read.
int refresh_wt(ofx_mlp* n) {
    for (int l = 0; l < NLAYER; ++l) OFX_TRY(transpose(n, n->wb[l], n->kin[l], n->kout[l], n->wt[l], n->kout[l]));
    return 0;
}

// Loss and gradients of n samples (rows idx of x, t; null: all of them), then
// an Adam step or the gradient vector.  The loss goes to loss.
int grad_step(ofx_mlp* n, const float* x, const float* t, const int* idx, int nsamp, bool adam, float lr, float* loss) {
    const int Mp = (nsamp + 63) / 64 * 64;
    MlpTrain T;
    for (int l = 0; l < NLAYER; ++l) {
        T.wf[l] = n->wf[l]; T.wb_frag[l] = n->wb_frag[l]; T.b[l] = n->b[l];
        T.hT[l] = n->hT[l]; T.gT[l] = n->gT[l]; T.cs[l] = n->cs[l];
    }
    T.lpart = n->lpart; T.x = x; T.t = t; T.idx = idx; T.n = nsamp; T.Mp = Mp;
    if (Mp <= 16 * 256) k_mlp_grad<1, 8, 8><<<Mp / 16, 512, 0, n->stream>>>(T);
    else k_mlp_grad<2, 8, 3><<<Mp / 32, 512, 0, n->stream>>>(T);
    OFX_HIP(hipGetLastError());
    MlpWgrad G;
    MlpUpdate U;
    const int ns = wgrad_splits(Mp);
    const bool together = ns <= SPLITS_TOGETHER;
    size_t o = 0;
    for (int l = 0; l < NLAYER; ++l) {
        G.hT[l] = n->hT[l]; G.gT[l] = n->gT[l];
        G.part[l] = n->part + o;
        if (together) o += (size_t)ns * wgrad_elems(l);
        U.w[l] = n->w[l]; U.m[l] = n->mw[l]; U.v[l] = n->vw[l]; U.b[l] = n->b[l]; U.mb[l] = n->mb[l]; U.vb[l] = n->vb[l];
        U.wb[l] = n->wb[l]; U.wf[l] = n->wf[l]; U.wb_frag[l] = n->wb_frag[l];
        U.part[l] = G.part[l]; U.cs[l] = n->cs[l];
    }
    G.Mp = Mp; G.ks = Mp / ns;
    U.lpart = n->lpart; U.grad = n->grad; U.loss = loss; U.nsplit = ns; U.Mp = Mp; U.n = nsamp;
    U.lr = lr; U.b1 = 0.9f; U.b2 = 0.999f; U.eps = 1e-8f; U.c1 = U.c2 = 0.f;
    if (adam) {
        ++n->step;
        U.c1 = 1.0f / (1.0f - std::pow(U.b1, (float)n->step));
        U.c2 = 1.0f / (1.0f - std::pow(U.b2, (float)n->step));
    }
    for (int l0 = 0; l0 < NLAYER; l0 = together ? NLAYER : l0 + 1) {
        const int l1 = together ? NLAYER : l0 + 1;
        int tiles = 0, blocks = l0 == 0 ? 1 : 0;
        for (int l = l0; l < l1; ++l) { tiles += wg_tm(l) * wg_tn(l); blocks += upd_wblocks(l) + upd_bblocks(l); }
        k_wgrad<<<dim3(tiles, ns), 256, 0, n->stream>>>(G, l0, l1);
        if (adam) k_update<true><<<blocks, 256, 0, n->stream>>>(U, l0, l1);
        else k_update<false><<<blocks, 256, 0, n->stream>>>(U, l0, l1);
    }
    OFX_HIP(hipGetLastError());
    return 0;
}

// ---- allocation-free forward pass (ofx_mlp_forward_noalloc)
// Its work arrays live in one file-scope device array, `scratch`, of a fixed
// size: packed inputs [MAXN][16] bf16, two activation buffers [MAXN][256]
// bf16 (layers alternate between them) and the padded outputs [MAXN][64]
// fp32 -- 10.25 MiB, held by every GPU the library runs on until the process
// ends.  Every call on one GPU uses that GPU's copy; each element a call reads
// it has written first, so nothing needs clearing, and calls that overlap on
// one GPU race.
constexpr int NOALLOC_MAXN = 8192;
constexpr size_t NOALLOC_IN = sizeof(bf16) * NOALLOC_MAXN * NIN_P;
constexpr size_t NOALLOC_ACT = sizeof(bf16) * NOALLOC_MAXN * NHID;
constexpr size_t NOALLOC_OUT = sizeof(float) * NOALLOC_MAXN * NOUT_P;
constexpr size_t NOALLOC_BYTES = NOALLOC_IN + 2 * NOALLOC_ACT + NOALLOC_OUT;
static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

std::mutex g_scratch_mu;
std::vector<unsigned char*> g_scratch_ptr;  // device id -> address of its `scratch`

// The device address of `scratch` on `device`, looked up once per device with
// that device current (host code must never pass the array's name itself).
int scratch_address(int device, unsigned char** out) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if ((int)g_scratch_ptr.size() <= device) g_scratch_ptr.resize(device + 1, nullptr);
    if (!g_scratch_ptr[device]) {
        int cur = 0;
        OFX_HIP(hipGetDevice(&cur));
        OFX_HIP(hipSetDevice(device));
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        (void)hipSetDevice(cur);
        if (e != hipSuccess || !p) {
            set_error(std::string("mlp: hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
            return OFX_EHIP;
        }
        g_scratch_ptr[device] = static_cast<unsigned char*>(p);
    }
    *out = g_scratch_ptr[device];
    return 0;
}

}  // namespace

extern "C" {

int ofx_mlp_create(ofx_mlp** out, int device, unsigned long long seed) {
    if (!out) { set_error("null out"); return OFX_EINVAL; }
    *out = nullptr;
    ofx_mlp* n = new (std::nothrow) ofx_mlp();
    if (!n) { set_error("out of host memory"); return OFX_ENOMEM; }
    n->device = device;
    int rc = 0;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) != hipSuccess) {
        set_error("mlp: no such HIP device");
        delete n;
        return OFX_EHIP;
    }
    for (int l = 0; l < NLAYER; ++l) {
        n->kin[l] = (l == 0) ? NIN_P : NHID;
        n->kout[l] = (l == NLAYER - 1) ? NOUT_P : NHID;
    }
    unsigned char* sp = nullptr;  // the allocation-free forward's work array on this device
    rc = scratch_address(device, &sp);
    if (!rc) { void* p; rc = mlp_alloc(n, &p, sizeof(float) * lay_off(NLAYER)); n->grad = (float*)p; }
    std::vector<float> hw, hb;
    uint64_t s = seed * 6364136223846793005ull + 1442695040888963407ull;
    auto urand = [&]() {  // uniform in [-1, 1)
        s = s * 6364136223846793005ull + 1442695040888963407ull;
        return (float)((double)(s >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0);
    };
    for (int l = 0; l < NLAYER && !rc; ++l) {
        size_t nw = (size_t)n->kin[l] * n->kout[l];
        int fan_in = (l == 0) ? NIN : NHID;
        int real_out = (l == NLAYER - 1) ? NOUT : NHID;
        float a = std::sqrt(6.0f / (float)fan_in);  // uniform He-style initialisation
        hw.assign(nw, 0.0f);
        for (int i = 0; i < ((l == 0) ? NIN : NHID); ++i)
            for (int j = 0; j < real_out; ++j) hw[(size_t)i * n->kout[l] + j] = a * urand();
        hb.assign(n->kout[l], 0.0f);
        void* p;
        rc = mlp_alloc(n, &p, sizeof(float) * nw); n->w[l] = (float*)p;
        if (!rc) { rc = mlp_alloc(n, &p, sizeof(float) * n->kout[l]); n->b[l] = (float*)p; }
        if (!rc) { rc = mlp_alloc(n, &p, sizeof(bf16) * nw); n->wb[l] = (bf16*)p; }
        if (!rc) { rc = mlp_alloc(n, &p, sizeof(bf16) * nw); n->wt[l] = (bf16*)p; }
        if (!rc) { rc = mlp_alloc(n, &p, sizeof(float) * nw); n->mw[l] = (float*)p; }
        if (!rc) { rc = mlp_alloc(n, &p, sizeof(float) * nw); n->vw[l] = (float*)p; }
        if (!rc) { rc = mlp_alloc(n, &p, sizeof(float) * n->kout[l]); n->mb[l] = (float*)p; }
        if (!rc) { rc = mlp_alloc(n, &p, sizeof(float) * n->kout[l]); n->vb[l] = (float*)p; }
        if (!rc) { rc = mlp_alloc(n, &p, sizeof(bf16) * 512 * frag_tiles(l) * frag_steps(l)); n->wf[l] = (bf16*)p; }
        if (!rc) { rc = mlp_alloc(n, &p, sizeof(bf16) * 512 * (NHID / 16) * (NHID / 32)); n->wb_frag[l] = (bf16*)p; }
        if (!rc && hipMemcpyAsync(n->w[l], hw.data(), sizeof(float) * nw, hipMemcpyHostToDevice, n->stream) != hipSuccess)
            rc = OFX_EHIP;
        if (!rc) {
            k_to_bf16<<<(unsigned)((nw + 255) / 256), 256, 0, n->stream>>>(n->w[l], nw, n->wb[l]);
            if (hipGetLastError() != hipSuccess) rc = OFX_EHIP;
        }
        if (!rc && hipStreamSynchronize(n->stream) != hipSuccess) rc = OFX_EHIP;
    }
    if (!rc) rc = refresh_wt(n);
    if (!rc) rc = refresh_frag(n);
    // (ofx_mlp_forward_noalloc may read them on any stream next)
    if (!rc && hipStreamSynchronize(n->stream) != hipSuccess) rc = OFX_EHIP;
    if (rc) {
        ofx_mlp_destroy(n);
        return rc;
    }
    *out = n;
    return 0;
}

int ofx_mlp_destroy(ofx_mlp* n) {
    if (!n) return 0;
    (void)hipSetDevice(n->device);
    if (n->stream) (void)hipStreamSynchronize(n->stream);
    for (void* p : n->allocs) (void)hipFree(p);
    for (void* p : n->fwd_allocs) (void)hipFree(p);
    if (n->io_x) (void)hipFree(n->io_x);
    if (n->tbuf) (void)hipFree(n->tbuf);
    for (hipEvent_t e : n->out_ready)
        if (e) (void)hipEventDestroy(e);
    if (n->out_stream) (void)hipStreamDestroy(n->out_stream);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
    return 0;
}

int ofx_mlp_param_count(ofx_mlp* n, int* count) {
    if (!n || !count) { set_error("null argument"); return OFX_EINVAL; }
    int c = 0;
    for (int l = 0; l < NLAYER; ++l) c += n->kin[l] * n->kout[l] + n->kout[l];
    *count = c;
    return 0;
}

// Parameters as one fp32 vector: for each layer W[kin_p][kout_p]
// then b[kout_p] (padded shapes: 16/256/.../256 -> 256/.../64).
static int mlp_copy(ofx_mlp* n, float* host, bool to_device) {
    for (int l = 0; l < NLAYER; ++l) {
        size_t nw = (size_t)n->kin[l] * n->kout[l], o = lay_off(l);
        if (to_device) {
            OFX_HIP(hipMemcpyAsync(n->w[l], host + o, sizeof(float) * nw, hipMemcpyHostToDevice, n->stream));
            OFX_HIP(hipMemcpyAsync(n->b[l], host + o + nw, sizeof(float) * n->kout[l], hipMemcpyHostToDevice, n->stream));
            k_to_bf16<<<(unsigned)((nw + 255) / 256), 256, 0, n->stream>>>(n->w[l], nw, n->wb[l]);
        } else {
            OFX_HIP(hipMemcpyAsync(host + o, n->w[l], sizeof(float) * nw, hipMemcpyDeviceToHost, n->stream));
            OFX_HIP(hipMemcpyAsync(host + o + nw, n->b[l], sizeof(float) * n->kout[l], hipMemcpyDeviceToHost, n->stream));
        }
    }
    if (to_device) {
        OFX_TRY(refresh_wt(n));
        OFX_TRY(refresh_frag(n));
    }
    OFX_HIP(hipStreamSynchronize(n->stream));
    return 0;
}

int ofx_mlp_get_params(ofx_mlp* n, float* host) {
    if (!n || !host) { set_error("null argument"); return OFX_EINVAL; }
    return mlp_copy(n, host, false);
}

int ofx_mlp_set_params(ofx_mlp* n, const float* host) {
    if (!n || !host) { set_error("null argument"); return OFX_EINVAL; }
    n->step = 0;
    return mlp_copy(n, const_cast<float*>(host), true);
}

int ofx_mlp_forward(ofx_mlp* n, const float* x, int nsamp, float* y) {
    if (!n || !x || !y || nsamp < 1 || nsamp > MLP_MAXN) { set_error("mlp_forward: bad arguments"); return OFX_EINVAL; }
    OFX_HIP(hipSetDevice(n->device));
    const size_t cnt = (size_t)nsamp * NOUT;
    if (n->fwd_variant == 1) {
        OFX_TRY(io_reserve(n, nsamp));
        if (nsamp >= PIPE_MIN && !overlapping(x, y, nsamp)) {
            const int rc = forward_piped(n, x, nsamp, y);
            if (rc != OFX_ESTATE) return rc;
        }
        OFX_HIP(hipMemcpyAsync(n->io_x, x, sizeof(float) * (size_t)nsamp * NIN, hipMemcpyHostToDevice, n->stream));
        OFX_TRY(forward_fused(n, n->stream, n->io_x, nsamp, n->io_y));
        OFX_HIP(hipMemcpyAsync(y, n->io_y, sizeof(float) * cnt, hipMemcpyDeviceToHost, n->stream));
    } else {
        OFX_TRY(layered_reserve(n, nsamp));
        const int Mp = (nsamp + 63) / 64 * 64;
        OFX_HIP(hipMemcpyAsync(n->xin, x, sizeof(float) * (size_t)nsamp * NIN, hipMemcpyHostToDevice, n->stream));
        k_pack_inputs<<<(Mp * NIN_P + 255) / 256, 256, 0, n->stream>>>(n->xin, nsamp, Mp, n->h[0]);
        OFX_TRY(forward_layered(n, n->stream, n->h[0], Mp, [&](int l) { return n->h[l + 1]; }, n->y));
        k_pack_outputs<<<(unsigned)((cnt + 255) / 256), 256, 0, n->stream>>>(n->y, nsamp, n->yd);
        OFX_HIP(hipGetLastError());
        OFX_HIP(hipMemcpyAsync(y, n->yd, sizeof(float) * cnt, hipMemcpyDeviceToHost, n->stream));
    }
    OFX_HIP(hipStreamSynchronize(n->stream));
    return 0;
}

int ofx_mlp_forward_noalloc(ofx_mlp* n, const float* x_dev, int nsamp, float* y_dev, void* stream) {
    if (!n || !x_dev || !y_dev || nsamp < 1) { set_error("mlp_forward_noalloc: bad arguments"); return OFX_EINVAL; }
    if (nsamp > NOALLOC_MAXN) {
        set_error("mlp_forward_noalloc: at most 8192 samples per call (fixed work array)");
        return OFX_EINVAL;
    }
    OFX_HIP(hipSetDevice(n->device));
    hipStream_t st = stream ? static_cast<hipStream_t>(stream) : n->stream;
    if (n->fwd_variant == 1 && !overlapping(x_dev, y_dev, nsamp)) return forward_fused(n, st, x_dev, nsamp, y_dev);
    unsigned char* base = nullptr;
    OFX_TRY(scratch_address(n->device, &base));
    if (n->fwd_variant == 1) {  // y_dev overwrites inputs: from a copy of them
        static_assert(sizeof(float) * NOALLOC_MAXN * NIN <= NOALLOC_BYTES, "room for the inputs");
        float* in = reinterpret_cast<float*>(base);
        k_copy_floats<<<(nsamp * NIN + 255) / 256, 256, 0, st>>>(x_dev, nsamp * NIN, in);
        OFX_HIP(hipGetLastError());
        return forward_fused(n, st, in, nsamp, y_dev);
    }
    bf16* in = reinterpret_cast<bf16*>(base);
    bf16* act[2] = {reinterpret_cast<bf16*>(base + NOALLOC_IN), reinterpret_cast<bf16*>(base + NOALLOC_IN + NOALLOC_ACT)};
    float* yp = reinterpret_cast<float*>(base + NOALLOC_IN + 2 * NOALLOC_ACT);
    const int Mp = (nsamp + 63) / 64 * 64;
    k_pack_inputs<<<(Mp * NIN_P + 255) / 256, 256, 0, st>>>(x_dev, nsamp, Mp, in);
    OFX_HIP(hipGetLastError());
    OFX_TRY(forward_layered(n, st, in, Mp, [&](int l) { return act[l & 1]; }, yp));
    size_t cnt = (size_t)nsamp * NOUT;
    k_pack_outputs<<<(unsigned)((cnt + 255) / 256), 256, 0, st>>>(yp, nsamp, y_dev);
    OFX_HIP(hipGetLastError());
    return 0;
}

int ofx_mlp_set_forward_variant(ofx_mlp* n, int variant) {
    if (!n || variant < 0 || variant > 1) { set_error("mlp_set_forward_variant: variant 0 or 1"); return OFX_EINVAL; }
    n->fwd_variant = variant;
    return 0;
}

int ofx_mlp_gradients(ofx_mlp* n, const float* x, const float* t, int nsamp, float* loss, float* grads) {
    if (!n || !x || !t || nsamp < 1 || nsamp > MLP_MAXN) { set_error("mlp_gradients: bad arguments"); return OFX_EINVAL; }
    OFX_HIP(hipSetDevice(n->device));
    OFX_TRY(train_reserve(n, nsamp));
    OFX_HIP(hipMemcpyAsync(n->tx, x, sizeof(float) * (size_t)nsamp * NIN, hipMemcpyHostToDevice, n->stream));
    OFX_HIP(hipMemcpyAsync(n->tt, t, sizeof(float) * (size_t)nsamp * NOUT, hipMemcpyHostToDevice, n->stream));
    OFX_TRY(grad_step(n, n->tx, n->tt, nullptr, nsamp, false, 0.f, n->loss));
    if (loss) OFX_HIP(hipMemcpyAsync(loss, n->loss, sizeof(float), hipMemcpyDeviceToHost, n->stream));
    if (grads) OFX_HIP(hipMemcpyAsync(grads, n->grad, sizeof(float) * lay_off(NLAYER), hipMemcpyDeviceToHost, n->stream));
    OFX_HIP(hipStreamSynchronize(n->stream));
    return 0;
}

int ofx_mlp_train(ofx_mlp* n, const float* x, const float* t, int nsamp, int batch, int steps, float lr,
                  unsigned long long seed, float* loss_out) {
    if (!n || !x || !t || nsamp < 1 || batch < 64 || batch > MLP_MAXN || steps < 1) {
        set_error("mlp_train: bad arguments");
        return OFX_EINVAL;
    }
    OFX_HIP(hipSetDevice(n->device));
    int bsz = std::min(batch, nsamp);
    OFX_TRY(train_reserve(n, bsz));
    // training set, epoch permutation and per-step losses live on the device
    float *dx = nullptr, *dt = nullptr, *dl = nullptr;
    int* dperm = nullptr;
    int rc = 0;
    if (hipMalloc(&dx, sizeof(float) * (size_t)nsamp * NIN) != hipSuccess ||
        hipMalloc(&dt, sizeof(float) * (size_t)nsamp * NOUT) != hipSuccess ||
        hipMalloc(&dperm, sizeof(int) * (size_t)nsamp) != hipSuccess ||
        hipMalloc(&dl, sizeof(float) * (size_t)steps) != hipSuccess) {
        set_error("mlp_train: out of device memory");
        rc = OFX_ENOMEM;
    }
    if (!rc && (hipMemcpyAsync(dx, x, sizeof(float) * (size_t)nsamp * NIN, hipMemcpyHostToDevice, n->stream) != hipSuccess ||
                hipMemcpyAsync(dt, t, sizeof(float) * (size_t)nsamp * NOUT, hipMemcpyHostToDevice, n->stream) != hipSuccess))
        rc = OFX_EHIP;
    std::vector<int> perm(nsamp);
    for (int i = 0; i < nsamp; ++i) perm[i] = i;
    uint64_t s = seed * 2862933555777941757ull + 3037000493ull;
    int pos = nsamp;
    for (int st = 0; st < steps && !rc; ++st) {
        if (pos + bsz > nsamp) {  // new epoch: reshuffle (Fisher-Yates) and upload
            for (int i = nsamp - 1; i > 0; --i) {
                s = s * 6364136223846793005ull + 1442695040888963407ull;
                int j = (int)((s >> 33) % (uint64_t)(i + 1));
                std::swap(perm[i], perm[j]);
            }
            if (hipStreamSynchronize(n->stream) != hipSuccess ||
                hipMemcpy(dperm, perm.data(), sizeof(int) * (size_t)nsamp, hipMemcpyHostToDevice) != hipSuccess) {
                rc = OFX_EHIP;
                break;
            }
            pos = 0;
        }
        rc = grad_step(n, dx, dt, dperm + pos, bsz, true, lr, dl + st);
        pos += bsz;
    }
    if (const int r2 = refresh_wt(n)) rc = rc ? rc : r2;
    if (!rc && hipStreamSynchronize(n->stream) != hipSuccess) rc = OFX_EHIP;
    if (!rc && loss_out && hipMemcpy(loss_out, dl, sizeof(float) * (size_t)steps, hipMemcpyDeviceToHost) != hipSuccess)
        rc = OFX_EHIP;
    if (rc == OFX_EHIP) set_error("mlp_train: HIP error");
    (void)hipStreamSynchronize(n->stream);
    if (dx) (void)hipFree(dx);
    if (dt) (void)hipFree(dt);
    if (dperm) (void)hipFree(dperm);
    if (dl) (void)hipFree(dl);
    return rc;
}

}  // extern "C"
