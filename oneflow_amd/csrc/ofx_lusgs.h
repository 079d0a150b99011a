// ofx_lusgs.h -- per-cell and per-face pieces of the NS LU-SGS sweeps, shared
// by the level kernels (ofx_ns.hip) and the pipelined sweeps (ofx_sweep.hip).
#pragma once

#include "ofx_physics.h"

namespace ofx {

// Time step after UTimeStep::ModifyTimeStep (codes/uns/src/UTimeStep.cpp:368-381)
// and the LU-SGS diagonal of UNsSpectrum::CalcImplicitSpectrum
// (codes/uns/src/UNsSpectrum.cpp:52-94, sp2 = 1), evaluated where consumed.
__device__ __forceinline__ double clamped_dt(const DevFields& d, const Consts& k, int i, double mindt) {
    double dt = d.timestep[i];
    if (k.max_time_ratio > 0) {
        double mp = k.max_time_ratio * mindt;
        dt = (dt < mp) ? dt : mp;
    }
    return dt;
}
__device__ __forceinline__ double ns_impsr(const DevMesh& m, const DevFields& d, const Consts& k, int i, double mindt) {
    double imp = (1.0 / clamped_dt(d, k, i, mindt)) * m.vol[i];
    imp += d.invsr[i];
    imp += d.vissr[i];
    return imp;
}

// What a face contributes to the sweep of cell i without the neighbour's
// increment: the split eigenvalues and the factors of UNsLusgs::Solve.
struct LuFace {
    double lmd1, x1, x2, c2, vn, af, hm, visrad;
};

// UNsLusgs::Solve for face f seen from cell i: GCom::SetGeometry orientation,
// PrepareData/PrepareDataFacePrim, NsLusgs::GetStandardFluxIncrement(-1) with
// CalcFaceEigenValue and CalcDH, then CalcViscousTerm and AddFluxIncrement
// (codes/uns/src/UNsLusgs.cpp:189-335, codes/ns/src/NsLusgs.cpp:121-228,340-368).
// The part that depends on the states alone, for cell i = l (after
// GCom::SetGeometry has put i on the left) and neighbour r.  Own state
// (rl..pl) and neighbour data are passed in, loaded by the caller.
// VM: the viscous term of the face, 0 none (inviscid), 1 spectral-radius
// model 1 (neighbour volume), 2 models 2 and 3 (centre distance) -- a
// compile-time choice, so a face evaluates only its own model.
template <int VM>
__device__ __forceinline__ LuFace ns_lusgs_coef(const Consts& k, double xfn, double yfn, double zfn, double vfn,
                                                double farea, double rl, double ul, double vl, double wl, double pl,
                                                const double* pj, double visl, double vist, double volr, double dist) {
    LuFace f;
    double rr = pj[0], ur = pj[1], vr = pj[2], wr = pj[3], pr = pj[4];
    double gl = k.gama, gr = k.gama;
    double hl = gl / (gl - 1.0) * pl / rl + 0.5 * sqr3(ul, vl, wl);
    double hr = gr / (gr - 1.0) * pr / rr + 0.5 * sqr3(ur, vr, wr);
    double tmp0 = sqrt(rr / rl);
    double tmp1 = 1.0 / (1.0 + tmp0);
    double rm = sqrt(rr * rl);
    double um = (ul + ur * tmp0) * tmp1;
    double vm = (vl + vr * tmp0) * tmp1;
    double wm = (wl + wr * tmp0) * tmp1;
    double hm = (hl + hr * tmp0) * tmp1;
    double pm = rm * (hm - 0.5 * sqr3(um, vm, wm)) * (gl - 1.0) / gl;
    double gama = k.gama;
    double c2f = dabs(gama * pm / rm);
    double cmf = sqrt(c2f);
    double vnf = xfn * um + yfn * vm + zfn * wm;
    double lmdF = dabs(vnf - vfn) + cmf;
    f.c2 = dabs(gama * pj[4] / pj[0]);
    double cm = sqrt(f.c2);
    f.vn = xfn * pj[1] + yfn * pj[2] + zfn * pj[3];
    double vn_rel = f.vn - vfn;
    f.lmd1 = 0.5 * (vn_rel + -1.0 * lmdF);
    double lmd2 = 0.5 * ((vn_rel + cm) + -1.0 * lmdF);
    double lmd3 = 0.5 * ((vn_rel - cm) + -1.0 * lmdF);
    f.x1 = (f.lmd1 + f.lmd1 - lmd2 - lmd3) / (f.c2 + f.c2);
    f.x2 = (lmd2 - lmd3) / (cm + cm);
    double v2 = sqr3(pj[1], pj[2], pj[3]);
    double ae = gama - 1.0;
    f.af = 0.5 * ae * v2;
    double enth = (gama / (gama - 1.0)) * (pj[4] / pj[0]);
    f.hm = enth + 0.5 * v2;
    f.visrad = 0.0;
    if (VM == 1) {
        double density = 0.5 * (rl + rr);
        double c1 = 4.0 / 3.0 * (visl + vist);
        double cc2 = k.gama * (visl * k.oprl + vist * k.oprt);
        double c3 = 2.0 * dmax(c1, cc2) / (k.reynolds * density);
        f.visrad = (farea * farea) * c3 / volr;
    } else if (VM == 2) {
        double viscosity = visl + vist;
        double density = 0.5 * (rl + rr);
        double c1 = 2.0 * viscosity / (density * dist * k.reynolds + SMALL);
        f.visrad = 0.5 * c1 * farea;
    }
    return f;
}

// The split flux increment dfj of the neighbour's dqj; returns the viscous radius
// (a sweep adds the face as rhs0 -= radius * dqj, then rhs0 += dfj).
template <int VM>
__device__ __forceinline__ double ns_lusgs_term(const Consts& k, double xfn, double yfn, double zfn, double vfn,
                                                double farea, double rl, double ul, double vl, double wl, double pl,
                                                const double* pj, const double* dqj, double visl, double vist,
                                                double volr, double dist, double* dfj) {
    const LuFace f = ns_lusgs_coef<VM>(k, xfn, yfn, zfn, vfn, farea, rl, ul, vl, wl, pl, pj, visl, vist, volr, dist);
    double dc = f.vn * dqj[0] - xfn * dqj[1] - yfn * dqj[2] - zfn * dqj[3];
    double c2dc = f.c2 * dc;
    double ae = k.gama - 1.0;
    double dh = -ae * (pj[1] * dqj[1] + pj[2] * dqj[2] + pj[3] * dqj[3] - dqj[4]);
    dh += f.af * dqj[0];
    double term1 = dh * f.x1 + dc * f.x2;
    double term2 = c2dc * f.x1 + dh * f.x2;
    dfj[0] = f.lmd1 * dqj[0] - term1;
    dfj[1] = f.lmd1 * dqj[1] - pj[1] * term1 + xfn * term2;
    dfj[2] = f.lmd1 * dqj[2] - pj[2] * term1 + yfn * term2;
    dfj[3] = f.lmd1 * dqj[3] - pj[3] * term1 + zfn * term2;
    dfj[4] = f.lmd1 * dqj[4] - f.hm * term1 + f.vn * term2;
    for (int e = 0; e < 5; ++e) dfj[e] *= farea;
    return f.visrad;
}

// The face term added to rhs0.
template <int VM>
__device__ __forceinline__ void ns_lusgs_face(const Consts& k, double xfn, double yfn, double zfn, double vfn,
                                              double farea, double rl, double ul, double vl, double wl, double pl,
                                              const double* pj, const double* dqj, double visl, double vist,
                                              double volr, double dist, double* rhs0) {
    double dfj[5];
    const double visrad = ns_lusgs_term<VM>(k, xfn, yfn, zfn, vfn, farea, rl, ul, vl, wl, pl, pj, dqj, visl, vist,
                                            volr, dist, dfj);
    if (VM != 0)
        for (int e = 0; e < 5; ++e) rhs0[e] -= visrad * dqj[e];
    for (int e = 0; e < 5; ++e) rhs0[e] += dfj[e];
}

// UNsUpdate::UpdateFlowField + NsUpdate::CalcFlowField / WeekSolutionFix
// (codes/uns/src/UNsUpdate.cpp:46-146, codes/ns/src/NsUpdate.cpp:40-67,192-217):
// the new primitive state of a cell; false when it needs SolutionFix.
__device__ __forceinline__ bool ns_update_state(const Consts& k, const double* prim0, const double* dq, double* prim) {
    double q0[5], q[5];
    double gama = k.gama;
    prim_to_q(prim0, gama, q0);
    for (int e = 0; e < 5; ++e) q[e] = q0[e] + dq[e];
    double density = dabs(q[0]);
    double rd = 1.0 / density;
    double um = q[1] * rd, vm = q[2] * rd, wm = q[3] * rd, rem = q[4];
    double v2 = sqr3(um, vm, wm);
    double reint = rem - 0.5 * density * v2;
    prim[0] = density; prim[1] = um; prim[2] = vm; prim[3] = wm; prim[4] = (gama - 1.0) * reint;
    if (prim[0] <= 0.0 || prim[4] <= 0.0) {
        const double coefs[3] = {0.5, 0.1, 0.01};
        for (int kk = 0; kk < 3; ++kk) {
            for (int e = 0; e < 5; ++e) prim[e] += coefs[kk] * dq[e];
            if (!(prim[0] < 0.0 || prim[4] < 0.0)) return true;
        }
        return false;
    }
    return true;
}

// A cell whose increment dq is final needs SolutionFix or not: if so, it raises the
// grid's flag (RQ_FIX) of parity `par`.  The update clears the other parity's.
__device__ __forceinline__ void ns_update_flag(const DevMesh& m, const DevFields& d, const Consts& k,
                                               const double* prim0, const double* dq, int par) {
    double prim[5];
    if (!ns_update_state(k, prim0, dq, prim))
        atomicMax(&d.slots[((size_t)par * m.nz * RQ_N + RQ_FIX) * NSLOT + blockIdx.x % NSLOT],
                  (unsigned long long)__double_as_longlong(1.0));
}

}  // namespace ofx
