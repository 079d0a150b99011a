// ofx_sweep.hip -- pipelined LU-SGS sweeps for numberings with many narrow
// dependency levels (structured-like orders; ofx_sweep.h has the schedule).
//
// Such a grid has hundreds of levels of a few dozen cells, each waiting for
// the one before, so a sweep's time is levels times the latency of one level.
// Launched level by level, a level costs a kernel of ~7 us; the pipelined sweep
// keeps one level's chain down to an LDS read, the increments' arithmetic and
// an LDS write by taking everything else out of it:
//   * one preparation kernel over all cells evaluates what the face terms hold
//     without the increments (square roots, divisions, eigenvalues) into
//     two streams, stored in the order each sweep walks the cells;
//   * a workgroup owns one range of cells and keeps its increments, and the
//     halo of earlier ranges' it needs, in LDS;
//   * its waves have one role each: loaders copy the stream ahead into an LDS
//     ring, one receiver polls the exchange buffer for halo increments, and
//     compute waves walk the levels.  NS takes 16 lanes per cell: a lane
//     computes one equation of every other face (after the two dot products
//     all equations share), and one division;
//   * a compute wave reads the next group's face terms while it works on the
//     current one, and divides by the stored reciprocal of the diagonal
//     (ofx_math.h, correctly rounded).
// Waves meet through counters in LDS (a wave's LDS operations complete in
// order, so a counter written after data is seen after it); no barrier.
//
// Ranges meet through the exchange buffer: the preparation kernel fills it
// with a signalling-NaN pattern no arithmetic produces, the owner stores each
// exported increment as one device-scope atomic, and the reader polls the
// value itself.  Workgroups take their range by a ticket drawn when they
// start, so a range's predecessors have always started before it: the first
// unfinished range never waits, whatever the dispatch order or the number of
// resident workgroups, and every wait ends.  As a guard a wave's waits also give
// up after sweep_polls polls, many times the longest chain.  No wave goes on as if
// it had been served: a loader stops (it overwrites nothing and publishes nothing, so
// that the compute waves give up in turn), the receiver hands out NaN for what it
// did not get, and a compute wave leaves NaN increments in the cells that it waited
// for in vain, which all that depend on them inherit and the residual norms report.
//
// The arithmetic is the level kernels' operation for operation.
//
// What bounds it: the latency of one level's chain, ~0.46 us NS and ~0.34 us SA
// (about 1100 and 800 cycles: one LDS round trip, 20 / 8 dependent FP64
// operations, the division), 0.6-1 us where levels are wider than a round or
// cells have three dependencies, and ~2 us per range the chain crosses.
// Measured, lower + upper sweep with the preparation, NS / SA in us:
//   RAE2822, 23,552 cells, 431 levels:      577 / 352 (one 1024-thread workgroup
//     walking all levels with a barrier between them: 9564 / 1188)
//   O-grid, 120,832 cells, 747 levels:     1355 / 655 (18645 / 2661)
//   plate, 960 cells, 63 levels:             80 (a launch per level: 862)
#include <algorithm>
#include <memory>
#include <new>
#include <vector>

#include "ofx_lusgs.h"
#include "ofx_sweep.h"

namespace ofx {

namespace {

typedef int sw_int4 __attribute__((ext_vector_type(4)));
typedef int sw_int2 __attribute__((ext_vector_type(2)));

constexpr unsigned long long SW_EMPTY = 0x7FF0A5A5DEADBEEFull;  // a signalling NaN: never a result of arithmetic
constexpr int SW_LDS = 160 * 1024;
// Most cells of a range, and cells per level it may hold.  Narrow ranges keep a
// level to one round of the compute waves; wide ones spare the chain handovers
// between ranges (~2 us), which pays where it crosses many: at 128 or more
// cells a level and at least as many levels as a level has cells (a front that is a
// line, not a surface).  us per step, 6 and 1024 / 16 and 2048: O-grids of 120,832
// cells and 747 levels 2240 / 2116, 168,000 and 879 2845 / 2704, 46,080 and 435
// 1315 / 1329, 15,360 and 247 790 / 1010; 150,000 quads and 799 1145 / 1068; 120,000
// triangles and 400 624 / 573; 30,720 quads and 367 497 / 817; 120,000 hexes and 148
// 597 / 803; 46,080 tets and 65 207 / 283.
struct RangeShape { int cells, width; };
inline RangeShape range_shape(int C, int nlev) {
    const int per = C / nlev;
    return per >= 128 && nlev >= per ? RangeShape{2048, 16} : RangeShape{1024, 6};
}

// Shapes per solver: NS 5 increments per cell, 16 lanes per cell; SA 1 and 1.
// CH cells per loader step, ring of 4 steps.
template <int NEQ>
struct Shape {
    static constexpr int LPC = NEQ == 5 ? 16 : 1;     // lanes per cell
    static constexpr int CPG = 64 / LPC;              // cells a compute wave handles at once
    static constexpr int NW = NEQ == 5 ? 3 : 2;       // compute waves (at most 3)
    static constexpr int NL = NEQ == 5 ? 4 : 3;       // loader waves
    static constexpr int WAVES = NW + 1 + NL;         // + the halo receiver
    static constexpr int CH = NEQ == 5 ? 16 : 64;
    static constexpr int NCH = 4, RC = CH * NCH;      // ring, cells
    static constexpr int IST = NEQ == 5 ? 6 : 1;      // doubles per cell of the increments in LDS
    // a stream cell: values[NEQ], diagonal, its reciprocal (0: divide), the
    // destination of the result and xid + 1 << 3 | dependencies; then the
    // dependencies' records
    static constexpr int HDR = NEQ == 5 ? 64 : 32;
    static constexpr int REC = NEQ == 5 ? 128 : 16;
    static constexpr int META = HDR - 8;
    static constexpr int stride(int ne) { return HDR + REC * ne; }
    static size_t lds(const SweepPlan& P, int groups, int ne) {
        return 32 + 8 * (size_t)((groups + 2) & ~1) + 8 * (size_t)(((P.R + P.maxHalo) * IST + 1) & ~1) +
               (size_t)RC * stride(ne);
    }
};

}  // namespace

// Device side of one sweep direction.
struct SweepDev {
    char *stream[2] = {nullptr, nullptr};  // NS, SA: cells in sweep order, Shape::stride bytes each
    unsigned long long* exch[2] = {nullptr, nullptr};
    int *posOf = nullptr, *rngOff = nullptr, *haloOff = nullptr, *haloX = nullptr;
    int* grpOff[2] = {nullptr, nullptr};      // NS, SA: the compute waves' lists (SweepGroups)
    SweepGroup* grp[2] = {nullptr, nullptr};
    int maxGrp[2] = {0, 0};
    SweepMeta* meta = nullptr;
    int* slot = nullptr;
    int C = 0, R = 0, W = 0, NE = 0, nX = 0, maxHalo = 0;
    int polls[2] = {0, 0};  // NS, SA: sweep_polls
};

struct SweepSet {
    SweepDev d[2];  // lower, upper
    int* ticket = nullptr;
    int NE = 0;  // records per stream cell, both directions
    size_t lds[2][2] = {{0, 0}, {0, 0}};  // [solver][direction]
    hipStream_t stream = nullptr;
    std::vector<void*> allocs;
    ~SweepSet() {
        if (!allocs.empty()) (void)hipStreamSynchronize(stream);
        for (void* p : allocs) (void)hipFree(p);
    }
};

namespace {

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// The static parts of the streams (SweepMeta, increment slots).
template <int NEQ>
__global__ void __launch_bounds__(256) k_sweep_init(SweepDev s, int NE, bool upper) {
    using S = Shape<NEQ>;
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= s.C) return;
    char* cell = s.stream[NEQ == 5 ? 0 : 1] + (size_t)p * S::stride(NE);
    const SweepMeta mt = s.meta[p];
    int* o = reinterpret_cast<int*>(cell + S::META);
    o[0] = upper ? mt.cell : mt.pos2;
    o[1] = (mt.xid + 1) << 3 | mt.n;
    for (int j = 0; j < s.NE; ++j)
        *reinterpret_cast<int*>(cell + S::HDR + S::REC * j + S::REC - 8) = s.slot[(size_t)p * s.NE + j];
}

__device__ __forceinline__ void sweep_reset(const SweepDev& lo, const SweepDev& up, int solver, int neq, int* ticket) {
    const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x, nt = (long)gridDim.x * blockDim.x;
    for (long t = tid; t < (long)lo.nX * neq; t += nt) lo.exch[solver][t] = SW_EMPTY;
    for (long t = tid; t < (long)up.nX * neq; t += nt) up.exch[solver][t] = SW_EMPTY;
    if (tid < 2) ticket[tid] = 0;
}

// NS preparation: every interior face term of every cell without its
// increment, the residual and the diagonal, into both streams.  A record is
// {lmd1, x1, x2, c2, af, area, visrad, u, v, w, hm, nx, ny, nz, vn, slot}.
// A block takes 64 cells: wave j evaluates entry j of their face lists (and j +
// PREP_W .. of long ones), a last wave the diagonals.  A thread that evaluated
// all faces of its cell was one long chain per wave with few waves: 960 cells
// 13.5 us, 23,552 cells 17.0 (now 6.4 and 10.9).
template <int MAXF>
constexpr int PREP_W = MAXF < 6 ? MAXF : 6;
template <int MAXF, int VM, bool EN>
__global__ void __launch_bounds__(64 * (PREP_W<MAXF> + 1)) k_sweep_prep_ns(DevMesh m, DevFields d, Consts k0, int par,
                                                                          SweepDev lo, SweepDev up, int NE,
                                                                          int* ticket) {
    using S = Shape<5>;
    constexpr int PW = PREP_W<MAXF>;
    sweep_reset(lo, up, 0, 5, ticket);
    const int w = uniform((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    const int i0 = xcd_block((int)gridDim.x) * 64 + lane;
    const bool live = i0 < m.C;
    const int i = live ? i0 : m.C - 1;  // every lane stays active for the wave reduction
    const int T = m.T;
    const Consts k = zoned(k0, m, cell_zone(m, i));
    const size_t st = (size_t)S::stride(NE);
    char* cl = lo.stream[0] + lo.posOf[i] * st;
    char* cu = up.stream[0] + up.posOf[i] * st;
    if (w == PW) {
        double mindt;
        wave_slot_result<1, false>(d.slots, par, m.nz * RQ_N, RQ_DTMIN, &mindt);
        const double rad = ns_impsr(m, d, k, i, zone_mindt(m, d, i, mindt));
        if (!live) return;
        double* vl5 = reinterpret_cast<double*>(cl);
        for (int e = 0; e < 5; ++e) vl5[e] = d.res[e * T + i];
        const double y = ofxm::div_reciprocal(rad);
        vl5[5] = rad;
        vl5[6] = y;
        reinterpret_cast<double*>(cu)[5] = rad;
        reinterpret_cast<double*>(cu)[6] = y;
        return;
    }
    const int n = m.c2fOff[i + 1] - m.c2fOff[i], lomask = m.lomask[i];
    int ent[MAXF];
#pragma unroll
    for (int j = 0; j < MAXF; ++j) ent[j] = (j < m.ellw) ? m.ellf[(size_t)j * m.C + i] : 0;
    int nbound = 0;  // boundary faces come first
#pragma unroll
    for (int j = 0; j < MAXF; ++j) nbound += j < n && ent[j] >= 0 && ent[j] < m.B;
    const double rl = d.q[i], ul = d.q[T + i], vl = d.q[2 * T + i], wl = d.q[3 * T + i], pl = d.q[4 * T + i];
    double xi = 0.0, yi = 0.0, zi = 0.0;
    if (VM == 2 && !EN) { xi = m.xcc[i]; yi = m.ycc[i]; zi = m.zcc[i]; }
#pragma unroll
    for (int j = 0; j < MAXF; ++j) {
        if (j % PW != w || !live || j >= n || j < nbound) continue;
        const int f = ent[j] >= 0 ? ent[j] : ~ent[j], r = m.elln[(size_t)j * m.C + i];
        double nx, ny, nz, ar;
        if (EN) {
            const dvec4 r4 = m.ellg[(size_t)(2 * m.ellw + j) * m.C + i];
            nx = r4.x; ny = r4.y; nz = r4.z; ar = r4.w;
        } else {
            nx = m.xfn[f]; ny = m.yfn[f]; nz = m.zfn[f]; ar = m.area[f];
        }
        double pj[5], visl = 0.0, vist = 0.0, volr = 0.0, dist = 0.0;
        for (int e = 0; e < 5; ++e) pj[e] = d.q[e * T + r];
        const bool own = ent[j] >= 0;  // GCom::SetGeometry: the normal points out of i
        if (!own) { nx = -nx; ny = -ny; nz = -nz; }
        const double vfn = own ? 0.0 : -0.0;
        if (VM != 0) {
            visl = d.visl[r]; vist = d.vist[r];
            if (VM == 1) volr = EN ? m.elldv[(size_t)(m.ellw + j) * m.C + i] : m.vol[r];
            else if (EN) dist = m.elldv[(size_t)j * m.C + i];
            else dist = dabs(nx * (m.xcc[r] - xi) + ny * (m.ycc[r] - yi) + nz * (m.zcc[r] - zi));
        }
        const LuFace c = ns_lusgs_coef<VM>(k, nx, ny, nz, vfn, ar, rl, ul, vl, wl, pl, pj, visl, vist, volr, dist);
        // the record's place: lower (upper) neighbours among the entries before it
        const int before = __popc(lomask & ((1 << j) - 1));
        const bool lower = (lomask >> j) & 1;
        dvec2* o = reinterpret_cast<dvec2*>((lower ? cl : cu) + S::HDR + S::REC * (lower ? before : j - nbound - before));
        o[0] = dvec2{c.lmd1, c.x1};
        o[1] = dvec2{c.x2, c.c2};
        o[2] = dvec2{c.af, ar};
        o[3] = dvec2{c.visrad, pj[1]};
        o[4] = dvec2{pj[2], pj[3]};
        o[5] = dvec2{c.hm, nx};
        o[6] = dvec2{ny, nz};
        reinterpret_cast<double*>(o)[14] = c.vn;
    }
}

// SA preparation: the off-diagonal face matrices in sweep order (matrix_l when
// the cell is the face's right cell, matrix_r otherwise; UTurbLusgs).
template <int MAXF>
__global__ void __launch_bounds__(256) k_sweep_prep_sa(DevMesh m, DevFields d, SweepDev lo, SweepDev up, int NE,
                                                       int* ticket) {
    using S = Shape<1>;
    sweep_reset(lo, up, 1, 1, ticket);
    const int i = xcd_block(gridDim.x) * 256 + threadIdx.x;
    if (i >= m.C) return;
    const int n = m.c2fOff[i + 1] - m.c2fOff[i];
    int ent[MAXF];
#pragma unroll
    for (int j = 0; j < MAXF; ++j) ent[j] = (j < m.ellw) ? m.ellf[(size_t)j * m.C + i] : 0;
    const int lomask = m.lomask[i];
    double mat[MAXF];
#pragma unroll
    for (int j = 0; j < MAXF; ++j) mat[j] = ent[j] >= 0 ? d.saface[2 * m.F + ent[j]] : d.saface[1 * m.F + ~ent[j]];
    const size_t st = (size_t)S::stride(NE);
    char* cl = lo.stream[1] + lo.posOf[i] * st;
    char* cu = up.stream[1] + up.posOf[i] * st;
    int nl = 0, nu = 0;
#pragma unroll
    for (int j = 0; j < MAXF; ++j) {
        const int f = ent[j] >= 0 ? ent[j] : ~ent[j];
        if (j >= n || f < m.B) continue;
        const bool lower = (lomask >> j) & 1;
        *reinterpret_cast<double*>((lower ? cl : cu) + S::HDR + S::REC * (lower ? nl : nu)) = mat[j];
        if (lower) ++nl; else ++nu;
    }
    const double rad = d.turbimpsr[i], y = ofxm::div_reciprocal(rad);
    *reinterpret_cast<dvec2*>(cl) = dvec2{d.turbres[i], rad};
    reinterpret_cast<double*>(cl)[2] = y;
    reinterpret_cast<double*>(cu)[1] = rad;
    reinterpret_cast<double*>(cu)[2] = y;
}

// The compiler keeps LDS accesses on their side (and loads counters anew); the
// hardware completes a wave's LDS operations in order.
#define SW_ORDER() asm volatile("" ::: "memory")

// The value of the lane eight up in the row of 16.
__device__ __forceinline__ double from_upper_half(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x108, 0xf, 0xf, false);  // row_shl:8
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x108, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// A compute wave's group: what a lane holds of its cell before the increments
// (NS: of every other dependency, from the first or second by its half).
template <int NEQ, int NE>
struct Group {
    static constexpr int NJ = NEQ == 5 ? (NE + 1) / 2 : NE;
    static constexpr int NR = NEQ == 5 ? 15 : 1;
    int dest, link;
    double val, rad, y;
    double r[NJ][NR], A[NJ], B[NJ];  // A, B: the factors of the lane's equation
    int sl[NJ];
};

// One sweep.  UPPER: the increment is dq + (-rhs0) / D with dq the lower
// sweep's (in the stream's values); otherwise (res - rhs0) / D, stored into
// the upper sweep's stream.  VISC: the NS face terms hold a viscous radius.
template <int NEQ, int NE, bool UPPER, bool VISC>
__global__ void __launch_bounds__(Shape<NEQ>::WAVES * 64) k_sweep_pipe(SweepDev s, char* stream2, double* dq, int T,
                                                                      double gama, int polls, int* ticket) {
    using S = Shape<NEQ>;
    constexpr int SV = NEQ == 5 ? 0 : 1;
    constexpr int NW = S::NW, NL = S::NL, CH = S::CH, NCH = S::NCH, RC = S::RC, IST = S::IST;
    constexpr int DONE = 0xffff;
    constexpr int st = S::stride(NE);
    extern __shared__ __align__(16) char sm[];
    // counters (16 bits each): ctr[0..2] the compute waves' current positions
    // (every cell before the smallest is done), ctr[3] halo increments
    // received, ctr[4] cells in the ring so far; then the range
    uint16_t* ctr = reinterpret_cast<uint16_t*>(sm);
    int* range = reinterpret_cast<int*>(sm + 16);
    sw_int2* grp = reinterpret_cast<sw_int2*>(sm + 32);
    double* inc = reinterpret_cast<double*>(sm + 32 + 8 * ((s.maxGrp[SV] + 2) & ~1));
    char* ring = reinterpret_cast<char*>(inc + (((s.R + s.maxHalo) * IST + 1) & ~1));
    const int t = threadIdx.x, w = uniform(t >> 6), lane = t & 63;
    if (t == 0) range[0] = atomicAdd(ticket, 1);
    if (t < 8) ctr[t] = t < NW || t == 3 || t == 4 ? 0 : DONE;
    __syncthreads();
    const int g = uniform(range[0]);
    const int p0 = s.rngOff[g], n = s.rngOff[g + 1] - p0;
    const int g0 = s.grpOff[SV][NW * g], g1 = s.grpOff[SV][NW * g + NW];
    for (int k = t; k < g1 - g0; k += S::WAVES * 64) grp[k] = reinterpret_cast<const sw_int2*>(s.grp[SV])[g0 + k];
    __syncthreads();
    const char* src = s.stream[SV] + (size_t)p0 * st;
    unsigned long long* exch = s.exch[SV];
    // one read of the counters, in scalar registers
    struct Ctr { int done, halo, ring; };
    auto counters = [&](const sw_int4& v) {
        const unsigned x = (unsigned)uniform(v.x), y = (unsigned)uniform(v.y), z = (unsigned)uniform(v.z);
        return Ctr{(int)min(min(x & 0xffffu, x >> 16), y & 0xffffu), (int)(y >> 16), (int)(z & 0xffffu)};
    };
    auto read_counters = [&]() {
        const sw_int4 v = *reinterpret_cast<const sw_int4*>(sm);
        SW_ORDER();
        return counters(v);
    };

    if (w > NW) {  // ---- loaders: chunk c = CH cells of the stream, contiguous
        constexpr int U = CH * st / 1024;  // 16-byte vectors per lane
        static_assert(CH * st % 1024 == 0, "whole vectors");
        int spin = 0;
        for (int c = w - NW - 1; c * CH < n; c += NL) {
            const sw_int4* a = reinterpret_cast<const sw_int4*>(src + (size_t)c * CH * st);
            sw_int4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = a[u * 64 + lane];
            // the chunk's ring slot is free once chunk c - NCH is consumed
            while (read_counters().done < (c - NCH + 1) * CH && ++spin < polls) __builtin_amdgcn_s_sleep(1);
            if (spin >= polls) return;
            sw_int4* o = reinterpret_cast<sw_int4*>(ring + (size_t)(c % NCH) * CH * st);
#pragma unroll
            for (int u = 0; u < U; ++u) o[u * 64 + lane] = v[u];
            SW_ORDER();
            while (read_counters().ring < c * CH && ++spin < polls) {}  // chunks are published in order
            if (spin >= polls) return;
            if (lane == 0) ctr[4] = (uint16_t)((c + 1) * CH);
            SW_ORDER();
        }
        return;
    }
    if (w == NW) {  // ---- halo receiver: one lane per item, published in order
        const int h0 = s.haloOff[g], nh = s.haloOff[g + 1] - h0;
        int spin = 0;
        for (int b = 0; b < nh; b += 64) {
            const int it = b + lane;
            bool wait = it < nh;
            const unsigned long long* a = exch + (size_t)(wait ? s.haloX[h0 + it] : 0) * NEQ;
            int seen = b;
            while (true) {
                if (wait) {
                    unsigned long long v[NEQ];
                    bool ok = true;
#pragma unroll
                    for (int e = 0; e < NEQ; ++e)
                        v[e] = __hip_atomic_load(a + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                    for (int e = 0; e < NEQ; ++e) ok = ok && v[e] != SW_EMPTY;
                    if (ok || spin >= polls) {
                        for (int e = 0; e < NEQ; ++e)
                            inc[(size_t)(s.R + it) * IST + e] =
                                ok ? __longlong_as_double((long long)v[e]) : __builtin_nan("");
                        wait = false;
                    }
                }
                const unsigned long long open = __ballot(wait);
                const int got = min(nh, b + (open ? __ffsll((long long)open) - 1 : 64));
                SW_ORDER();
                if (got > seen && lane == 0) ctr[3] = (uint16_t)got;
                SW_ORDER();
                seen = max(seen, got);
                if (!open) break;
                ++spin;
            }
        }
        return;
    }
    // ---- compute waves
    __builtin_amdgcn_s_setprio(2);
    const int c = lane / S::LPC, e = NEQ == 5 ? min(lane & 7, 4) : 0;
    const int half = NEQ == 5 ? (lane >> 3) & 1 : 0;  // NS: first or second of each pair of dependencies
    const bool lead = NEQ == 5 ? (lane & 15) < 5 : true;
    const double ae = gama - 1.0;
    using Grp = Group<NEQ, NE>;
    constexpr int NJ = Grp::NJ;
    int i = s.grpOff[SV][NW * g + w] - g0;
    const int i1 = s.grpOff[SV][NW * g + w + 1] - g0;
    int spin = 0;
    // the current group: cells [pos, pos + cnt) of a level that starts at
    // `start` and needs `need` halo items
    int pos = DONE, cnt = 0, start = 0, need = 0;
    auto unpack = [&](const sw_int2& x) {
        const unsigned a = (unsigned)uniform(x.x), b = (unsigned)uniform(x.y);
        pos = (int)(a & 0xffffu);
        cnt = (int)(a >> 16);
        start = (int)(b & 0xffffu);
        need = (int)(b >> 16);
    };
    auto load = [&](Grp& G) {  // the current group's terms (from wherever the ring stands, if not there yet)
        const char* cell = ring + (size_t)((pos + min(c, max(cnt - 1, 0))) & (RC - 1)) * st;
        const double* h = reinterpret_cast<const double*>(cell);
        G.dest = reinterpret_cast<const int*>(cell + S::META)[0];
        G.link = reinterpret_cast<const int*>(cell + S::META)[1];
        G.val = h[e];
        G.rad = h[NEQ];
        G.y = h[NEQ + 1];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int jj = NEQ == 5 ? min(2 * j + half, NE - 1) : j;
            const double* rec = reinterpret_cast<const double*>(cell + S::HDR + S::REC * jj);
#pragma unroll
            for (int u = 0; u < Grp::NR; ++u) G.r[j][u] = rec[u];
            if constexpr (NEQ == 5) {
                G.A[j] = rec[6 + e];   // u, v, w, hm (0: unused)
                G.B[j] = rec[10 + e];  // nx, ny, nz, vn (0: unused)
            }
            G.sl[j] = reinterpret_cast<const int*>(rec)[S::REC / 4 - 2];
        }
    };
    bool loaded = false;
    // One group, its terms in G if `loaded`.  The next group's terms are read
    // into N meanwhile; `loaded` then tells whether the ring held them.
    auto step = [&](Grp& G, Grp& N) {
        if (__builtin_expect(!loaded, 0)) {
            while (read_counters().ring < pos + cnt && ++spin < polls) {}
            load(G);
            if (spin >= polls) {  // given up: what the stores below need comes from memory, the value is NaN
                G.val = __builtin_nan("");
                const int* h = reinterpret_cast<const int*>(src + (size_t)(pos + min(c, cnt - 1)) * st + S::META);
                G.dest = h[0];
                G.link = h[1] & ~7;
            }
        }
        const int nd = G.link & 7;
        // The increments, once every cell of the earlier levels and the level's
        // halo items are there: counters and, behind them, increments are
        // read together; if a counter was short, the increments are read again.
        double qd[NJ][NEQ], qe[NJ];
        auto increments = [&]() {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const double* a = inc + ((NEQ == 5 ? 2 * j + half : j) < nd ? G.sl[j] : 0) * IST;
#pragma unroll
                for (int v = 0; v < NEQ; ++v) qd[j][v] = a[v];
                qe[j] = NEQ == 5 ? a[e] : qd[j][0];
            }
        };
        sw_int4 kv = *reinterpret_cast<const sw_int4*>(sm);
        SW_ORDER();
        increments();
        const sw_int2 nx = grp[i + 1];
        asm volatile("" : "+v"(kv) : : "memory");  // the counters are looked at with all reads under way
        const Ctr k = counters(kv);
        if (k.done < start || k.halo < need) {
            Ctr q;
            do { q = read_counters(); } while ((q.done < start || q.halo < need) && ++spin < polls);
            increments();
            SW_ORDER();
            if (__builtin_expect(spin >= polls, 0)) {  // given up; behind the reads and as a branch: a select before
                SW_ORDER();                            // them took 1-3 % of a sweep (3,410 quads: 223 against 217 us)
                G.val = __builtin_nan("");
            }
        }
        const int here = pos, ncell = cnt;
        ++i;
        unpack(nx);
        if (i >= i1) { pos = DONE; cnt = 0; }
        loaded = k.ring >= pos + cnt;
        load(N);
        double rhs = 0.0;
        if constexpr (NEQ == 5) {
            double vq[NJ], df[NJ];
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const double lmd1 = G.r[j][0], x1 = G.r[j][1], x2 = G.r[j][2], c2 = G.r[j][3], af = G.r[j][4],
                             ar = G.r[j][5], vr = G.r[j][6], u = G.r[j][7], v = G.r[j][8], ww = G.r[j][9],
                             fx = G.r[j][11], fy = G.r[j][12], fz = G.r[j][13], vn = G.r[j][14];
                const double* q = qd[j];
                double dc = vn * q[0] - fx * q[1] - fy * q[2] - fz * q[3];
                double c2dc = c2 * dc;
                double dh = -ae * (u * q[1] + v * q[2] + ww * q[3] - q[4]);
                dh += af * q[0];
                double term1 = dh * x1 + dc * x2;
                double term2 = c2dc * x1 + dh * x2;
                double f = lmd1 * qe[j] - (e == 0 ? term1 : G.A[j] * term1);
                const double f2 = f + G.B[j] * term2;
                f = e == 0 ? f : f2;
                df[j] = f * ar;
                vq[j] = VISC ? vr * qe[j] : 0.0;
            }
            // the sums in face order, on the cell's lower half
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                double nr = VISC ? rhs - vq[j] : rhs;
                nr += df[j];
                rhs = 2 * j < nd ? nr : rhs;
                if (2 * j + 1 < NE) {
                    const double v1 = VISC ? from_upper_half(vq[j]) : 0.0, f1 = from_upper_half(df[j]);
                    nr = VISC ? rhs - v1 : rhs;
                    nr += f1;
                    rhs = 2 * j + 1 < nd ? nr : rhs;
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const double nr = rhs + G.r[j][0] * qe[j];
                rhs = j < nd ? nr : rhs;
            }
        }
        const double num = UPPER ? -rhs : G.val - rhs;
        double x = ofxm::div_by(num, G.rad, G.y);
        if (__builtin_expect(!__all(ofxm::div_by_ok(num, G.y)), 0)) x = num / G.rad;
        if (UPPER) x = G.val + x;
        if (lead && c < ncell) {
            inc[(here + c) * IST + e] = x;
            if (UPPER) dq[(size_t)e * T + G.dest] = x;
            else reinterpret_cast<double*>(stream2 + (size_t)G.dest * st)[e] = x;
            if (G.link >> 3)
                __hip_atomic_store(exch + (size_t)((G.link >> 3) - 1) * NEQ + e,
                                   (unsigned long long)__double_as_longlong(x), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        SW_ORDER();
        if (lane == 0) ctr[w] = (uint16_t)pos;
        SW_ORDER();
    };
    if (i < i1) unpack(grp[i]);
    if (lane == 0) ctr[w] = (uint16_t)pos;
    SW_ORDER();
    Grp GA, GB;
    while (i < i1) {
        step(GA, GB);
        if (i >= i1) break;
        step(GB, GA);
    }
}

template <int NEQ, int NE, bool VISC>
int sweep_pair(ofx_ctx* c, SweepSet& s, double* dq) {
    using S = Shape<NEQ>;
    constexpr int sv = NEQ == 5 ? 0 : 1;
    const int set = c->sweep_polls;
    k_sweep_pipe<NEQ, NE, false, VISC><<<s.d[0].W, S::WAVES * 64, s.lds[sv][0], c->stream>>>(
        s.d[0], s.d[1].stream[sv], dq, c->m.T, c->k.gama, set ? set : s.d[0].polls[sv], s.ticket);
    k_sweep_pipe<NEQ, NE, true, VISC><<<s.d[1].W, S::WAVES * 64, s.lds[sv][1], c->stream>>>(
        s.d[1], nullptr, dq, c->m.T, c->k.gama, set ? set : s.d[1].polls[sv], s.ticket + 1);
    OFX_HIP(hipGetLastError());
    return 0;
}

template <int NEQ, bool VISC>
int sweep_pair_ne(ofx_ctx* c, SweepSet& s, double* dq) {
    switch (s.NE) {
        case 1:
        case 2: return sweep_pair<NEQ, 2, VISC>(c, s, dq);
        case 3: return sweep_pair<NEQ, 3, VISC>(c, s, dq);
        case 4: return sweep_pair<NEQ, 4, VISC>(c, s, dq);
        default: return sweep_pair<NEQ, SW_MAXNE, VISC>(c, s, dq);
    }
}

template <int MAXF, int VM>
void prep_ns(ofx_ctx* c, SweepSet& s) {
    const int nb = (c->m.C + 63) / 64, nt = 64 * (PREP_W<MAXF> + 1);
    if (c->normal_variant == 1)
        k_sweep_prep_ns<MAXF, VM, true><<<nb, nt, 0, c->stream>>>(c->m, c->d, c->k, c->par_dt, s.d[0], s.d[1], s.NE, s.ticket);
    else
        k_sweep_prep_ns<MAXF, VM, false><<<nb, nt, 0, c->stream>>>(c->m, c->d, c->k, c->par_dt, s.d[0], s.d[1], s.NE, s.ticket);
}
template <int MAXF>
void prep_ns_vm(ofx_ctx* c, SweepSet& s) {
    if (c->k.vismodel == 0) prep_ns<MAXF, 0>(c, s);
    else if (c->k.visSRModel == 1) prep_ns<MAXF, 1>(c, s);
    else prep_ns<MAXF, 2>(c, s);
}

template <int NEQ, int NE>
bool lds_limit() {
    const void* f[4] = {(const void*)k_sweep_pipe<NEQ, NE, false, false>, (const void*)k_sweep_pipe<NEQ, NE, true, false>,
                        (const void*)k_sweep_pipe<NEQ, NE, false, true>, (const void*)k_sweep_pipe<NEQ, NE, true, true>};
    for (int k = 0; k < (NEQ == 5 ? 4 : 2); ++k)
        if (hipFuncSetAttribute(f[k], hipFuncAttributeMaxDynamicSharedMemorySize, SW_LDS) != hipSuccess) return false;
    return true;
}

}  // namespace

int pipelined_lusgs_ns(ofx_ctx* c) {
    SweepSet& s = *c->sweep;
    const int mf = c->m.maxFacesPerCell;
    if (mf <= 4) prep_ns_vm<4>(c, s);
    else if (mf <= 6) prep_ns_vm<6>(c, s);
    else prep_ns_vm<16>(c, s);
    OFX_HIP(hipGetLastError());
    return c->k.vismodel == 0 ? sweep_pair_ne<5, false>(c, s, c->d.dq) : sweep_pair_ne<5, true>(c, s, c->d.dq);
}

int pipelined_lusgs_sa(ofx_ctx* c) {
    SweepSet& s = *c->sweep;
    const int mf = c->m.maxFacesPerCell, nb = (c->m.C + 255) / 256;
    if (mf <= 4) k_sweep_prep_sa<4><<<nb, 256, 0, c->stream>>>(c->m, c->d, s.d[0], s.d[1], s.NE, s.ticket);
    else if (mf <= 6) k_sweep_prep_sa<6><<<nb, 256, 0, c->stream>>>(c->m, c->d, s.d[0], s.d[1], s.NE, s.ticket);
    else k_sweep_prep_sa<16><<<nb, 256, 0, c->stream>>>(c->m, c->d, s.d[0], s.d[1], s.NE, s.ticket);
    OFX_HIP(hipGetLastError());
    return sweep_pair_ne<1, false>(c, s, c->d.turbdq);
}

// Whether a grid of C cells and nlev levels per sweep is swept by the pipeline.
// A level launched by itself takes ~7 us (NS) and ~3.9 us (SA) while it is
// narrow, and its share of the memory bandwidth when it is wide; the
// pipeline takes ~0.5 us per level plus ~600 cells per us (one workgroup per
// CU).  Measured NS pairs, level by level / pipelined: 70 levels of 198 hexes
// 1888 / 302 us, 63 levels of 15 quads 862 / 89, 33 levels of 9000 prisms and
// tets 649 / 1068; the lines cross near 3000 cells per level.  A colouring's
// few levels stay with their launches (the first is fused into the residual).
static bool use_pipeline(int C, int nlev) { return nlev > 8 && C / nlev < 3000; }

// Device memory of the schedule; OFX_ENOMEM leaves no error behind.
static int sweep_alloc(ofx_ctx* c, SweepSet& s, void** p, size_t bytes) {
    s.allocs.push_back(nullptr);
    if (hipMalloc(p, std::max<size_t>(bytes, 8)) != hipSuccess) {
        (void)hipGetLastError();
        return OFX_ENOMEM;
    }
    s.allocs.back() = *p;
    OFX_HIP(hipMemsetAsync(*p, 0, std::max<size_t>(bytes, 8), c->stream));
    return 0;
}

static int build_set(ofx_ctx* c, const MeshLists& lists) {
    const std::vector<int>&off = lists.off, &nb = lists.nb, &id = lists.id;
    const int C = c->m.C;
    const int nlev = std::max(c->m.nLevLo, c->m.nLevUp);
    if (!use_pipeline(C, nlev) || c->m.maxFacesPerCell > 16) return 0;
    std::vector<int> level[2] = {std::vector<int>(C), std::vector<int>(C)};  // by storage cell
    for (int sc = 0; sc < C; ++sc) { level[0][sc] = lists.lev[id[sc]]; level[1][sc] = lists.levU[id[sc]]; }
    // dependencies per cell in either direction, which size the ring
    int ne = 1;
    for (int sc = 0; sc < C; ++sc) {
        int lo = 0, up = 0;
        for (int k = off[sc]; k < off[sc + 1]; ++k)
            if (nb[k] < C) ++(id[nb[k]] < id[sc] ? lo : up);
        ne = std::max(ne, std::max(lo, up));
    }
    if (ne > SW_MAXNE || C >= 1 << 28) return 0;
    const int NE = ne <= 2 ? 2 : ne <= 4 ? ne : SW_MAXNE;
    // the largest ranges whose increments, groups and ring fit in LDS
    SweepPlan P[2];
    SweepGroups G[2][2];  // [direction][solver]
    const RangeShape shape = range_shape(C, nlev);
    for (int k = 0; k < 2; ++k) {
        bool fits = false;
        for (int R = shape.cells; R >= SW_RMIN && !fits; R = R * 3 / 4) {
            if (!build_sweep_plan(C, off, nb, id, level[k], k == 1, R, shape.width, P[k])) return 0;
            G[k][0] = sweep_groups(P[k], Shape<5>::CPG, Shape<5>::NW);
            G[k][1] = sweep_groups(P[k], Shape<1>::CPG, Shape<1>::NW);
            fits = Shape<5>::lds(P[k], G[k][0].max, NE) <= (size_t)SW_LDS &&
                   Shape<1>::lds(P[k], G[k][1].max, NE) <= (size_t)SW_LDS;
        }
        if (!fits || !sweep_polls(P[k], G[k][0]) || !sweep_polls(P[k], G[k][1])) return 0;
    }
    for (int k = 0; k < 2; ++k)
        for (int p = 0; p < C; ++p) P[k].meta[p].pos2 = P[1 - k].posOf[P[k].meta[p].cell];
    // (the attribute belongs to the current device)
    const bool ok = lds_limit<5, 2>() && lds_limit<5, 3>() && lds_limit<5, 4>() && lds_limit<5, SW_MAXNE>() &&
                    lds_limit<1, 2>() && lds_limit<1, 3>() && lds_limit<1, 4>() && lds_limit<1, SW_MAXNE>();
    if (!ok) return 0;
    std::unique_ptr<SweepSet> s(new (std::nothrow) SweepSet());
    if (!s) return OFX_ENOMEM;
    s->NE = NE;
    s->stream = c->stream;
    auto A = [&](void** p, size_t bytes) { return sweep_alloc(c, *s, p, bytes); };
    for (int k = 0; k < 2; ++k) {
        SweepDev& d = s->d[k];
        const SweepPlan& p = P[k];
        d.C = C; d.R = p.R; d.W = p.W; d.NE = p.NE; d.nX = p.nX; d.maxHalo = p.maxHalo;
        s->lds[0][k] = Shape<5>::lds(p, G[k][0].max, NE);
        s->lds[1][k] = Shape<1>::lds(p, G[k][1].max, NE);
        // streams: room for the last chunk's reads past the end
        OFX_TRY(A((void**)&d.stream[0], ((size_t)C + Shape<5>::CH) * Shape<5>::stride(NE)));
        OFX_TRY(A((void**)&d.stream[1], ((size_t)C + Shape<1>::CH) * Shape<1>::stride(NE)));
        OFX_TRY(A((void**)&d.exch[0], sizeof(double) * 5 * (size_t)std::max(1, p.nX)));
        OFX_TRY(A((void**)&d.exch[1], sizeof(double) * (size_t)std::max(1, p.nX)));
        auto put = [&](void** dst, const void* src, size_t bytes) -> int {
            OFX_TRY(A(dst, bytes));
            return upload(c, *dst, src, bytes);
        };
        OFX_TRY(put((void**)&d.posOf, p.posOf.data(), sizeof(int) * p.posOf.size()));
        OFX_TRY(put((void**)&d.rngOff, p.rngOff.data(), sizeof(int) * p.rngOff.size()));
        for (int v = 0; v < 2; ++v) {
            OFX_TRY(put((void**)&d.grpOff[v], G[k][v].off.data(), sizeof(int) * G[k][v].off.size()));
            OFX_TRY(put((void**)&d.grp[v], G[k][v].g.data(), sizeof(SweepGroup) * G[k][v].g.size()));
            d.maxGrp[v] = G[k][v].max;
            d.polls[v] = sweep_polls(p, G[k][v]);
        }
        OFX_TRY(put((void**)&d.haloOff, p.haloOff.data(), sizeof(int) * p.haloOff.size()));
        OFX_TRY(put((void**)&d.haloX, p.haloX.data(), sizeof(int) * p.haloX.size()));
        OFX_TRY(put((void**)&d.meta, p.meta.data(), sizeof(SweepMeta) * p.meta.size()));
        OFX_TRY(put((void**)&d.slot, p.slot.data(), sizeof(int) * p.slot.size()));
        k_sweep_init<5><<<(C + 255) / 256, 256, 0, c->stream>>>(d, NE, k == 1);
        k_sweep_init<1><<<(C + 255) / 256, 256, 0, c->stream>>>(d, NE, k == 1);
        OFX_HIP(hipGetLastError());
    }
    OFX_TRY(A((void**)&s->ticket, 2 * sizeof(int)));
    c->sweep = s.release();
    return 0;
}

// Build the pipelined schedule of a mesh that profits from it (at the mesh
// upload, once everything else is allocated; c->sweep stays empty otherwise and
// the level kernels run).  Its streams take 0.7 to 1.9 KB per cell (two to six
// dependencies); a mesh that leaves no memory for them is swept level by level,
// and they are given back when a later allocation needs the room (alloc_bytes).
int sweep_build(ofx_ctx* c, const MeshLists& lists) {
    sweep_free(c);  // of a mesh whose upload failed later on
    int rc;
    try {
        rc = build_set(c, lists);
    } catch (const std::bad_alloc&) {
        rc = OFX_ENOMEM;
    }
    return rc == OFX_ENOMEM ? 0 : rc;
}

void sweep_free(ofx_ctx* c) {
    delete c->sweep;
    c->sweep = nullptr;
}

}  // namespace ofx
