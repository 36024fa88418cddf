// swe_rows.h -- device helpers shared by the row kernels (swe_kernels.hip: one slice per wave, neighbours
// gathered from memory; swe_tiles.hip: one tile per workgroup, neighbours staged in LDS).
#pragma once
#include <hip/hip_runtime.h>

#include "swe_amd.h"
#include "swe_kernels.h"

namespace swe {
namespace {

enum SmbKind : int { SMB_ROUNDOFF = 0, SMB_2 = 1, SMB_1 = 2, SMB_GALERKIN = 3 };

constexpr double kPi = 3.141592653589793;   // ACOS(-1.d0)

// Slice of this wave: the waves of a launch take the listed slices in order (remap: XCD-aware
// workgroup order), one slice each; -1 past the end of the list.  The value (and everything
// derived from it: the instance, its constants, dt) is wave-uniform and kept in scalar registers;
// the lane's row is slice*64 + lane.
template <int BS>
__device__ __forceinline__ int wave_slice(const Mesh& M, int remap) {
    const int b = remap ? xcd_block() : (int)blockIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(b * (BS / 64) + (int)(threadIdx.x >> 6));
    if (w >= M.nact) return -1;
    return __builtin_amdgcn_readfirstlane(M.act[w]);
}

// Instance owning a slice; -1 for a free slice.
__device__ __forceinline__ int slice_inst(const Mesh& M, int slice) {
    return __builtin_amdgcn_readfirstlane(M.sl[slice].inst);
}

__device__ __forceinline__ int lane_of() { return (int)(threadIdx.x & 63); }

__device__ __forceinline__ bool takes_steps(const InstDev& D, int flags) {
    return D.state == INST_RUNNING && flags == 0 && D.time < D.tfinal && D.steps < D.max_steps;
}

__device__ __forceinline__ int64_t row_base(const Mesh& M, int i) {
    return M.sl[i >> 6].sbase + (i & 63);
}

// Per-entry arrays streamed once per pass (c_ij, the first-order viscosities; with SWE_NT_LOADS >= 2
// also the dt pass's d_ij): their loads and stores carry the non-temporal hint, so they do not
// displace the gathered node data from the caches (measured: 14.86 -> 14.70 ms per 16.8M-node step).
// SWE_NT_NODE: the same hint on the low-order solution (1: discharge, 2: depth too), written by
// k_fct_lo and read back only at the row itself.
#ifndef SWE_NT_NODE
#define SWE_NT_NODE 2
#endif
#ifndef SWE_NT_LOADS
#define SWE_NT_LOADS 2
#endif
typedef double dvec2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double2 ld_entry(const double2* p) {
#if SWE_NT_LOADS
    const dvec2 v = __builtin_nontemporal_load((const dvec2*)p);
    return make_double2(v.x, v.y);
#else
    return *p;
#endif
}
__device__ __forceinline__ double ld_entry1(const double* p) {
#if SWE_NT_LOADS > 1
    return __builtin_nontemporal_load(p);
#else
    return *p;
#endif
}
__device__ __forceinline__ void st_entry1(double* p, double v) {
#if SWE_NT_LOADS > 1
    __builtin_nontemporal_store(v, p);
#else
    *p = v;
#endif
}
__device__ __forceinline__ void st_entry(double2* p, double2 v) {
#if SWE_NT_LOADS
    dvec2 w;
    w.x = v.x;
    w.y = v.y;
    __builtin_nontemporal_store(w, (dvec2*)p);
#else
    *p = v;
#endif
}

// Column of slot p of row i: a 16-bit offset from the row (half the bytes of the 32-bit column,
// which is read only where the offset does not fit).
__device__ __forceinline__ int col_at(const Mesh& M, int64_t p, int i) {
    const int d = M.dcol[p];
    return (d != kColFar) ? i + d : M.col[p];
}

__device__ __forceinline__ void raise_flag(int* flags, int inst, int f) {
    if (f) atomicOr(flags + inst, f);
}

// LDS of one wave for the compacted lambda phase: per-row one_over_h and SQRT(g*ABS(h)), then
// one double per slot of the slice (slot offset q*64 + lane).
__device__ __forceinline__ double* wave_lds(double* smem, int wmax) {
    return smem + (size_t)(threadIdx.x >> 6) * (size_t)(2 + wmax) * 64;
}

// RK combination of SOURCES/main.f90:83,89 (stage 0 keeps the Euler output)
__device__ __forceinline__ double rk_combine(int stage, double uo, double ui) {
    if (stage == 1) return (3.0 * uo + ui) / 4.0;
    if (stage == 2) return (uo + 2.0 * ui) / 3.0;
    return ui;
}

// Source terms of one node, dispatched on type_test (update.f90:614-623): friction (425-452),
// my_friction (454-469), coriolis (471-486).  v1, v2 = velocity at U.  src is uniform per wave.
// Launches whose instances have no source term use the HAS_SRC = false kernels, which leave it out.
template <bool HAS_SRC>
__device__ __forceinline__ void add_sources(int src, const Node& I, double mi, double v1, double v2, double dt,
                                            const Consts& K, double& r2, double& r3) {
    if constexpr (!HAS_SRC) return;
    if (src == SRC_MANNING) {
        const double hs = pow43(fmaxF(I.h, K.htiny));
        const double vel = K.fric * sqrt_rn(v1 * v1 + v2 * v2);
        const double hloc = 1.0 * vel * dt;
        const double den = hs + fmaxF(hs, hloc);
        r2 = r2 - mi * I.qx * vel * 2.0 / den;
        r3 = r3 - mi * I.qy * vel * 2.0 / den;
    } else if (src == SRC_LINEAR) {
        r2 = r2 - mi * 0.2 * I.qx;
        r3 = r3 - mi * 0.2 * I.qy;
    } else if (src == SRC_CORIOLIS) {
        const double f = 2.0;
        r2 = r2 + mi * f * I.qy;
        r3 = r3 - mi * f * I.qx;
    }
}

// compute_dij of one off-diagonal entry from c_ij itself: the norm and the unit vector are
// evaluated with compute_dij's expressions (SOURCES/update.f90:306-310; correctly rounded sqrt and
// division, so the bits are the reference's), which costs a square root and two divisions per entry
// instead of storing 24 bytes of normal and norm per entry (measured faster in every pass).
__device__ __forceinline__ double dij_from_c(const double2 c, const Node& I, const Node& J, double ovh_i,
                                             double ovh_j, double sql, double sqr, const Consts& K,
                                             const Rcp& r16, int& err) {
    const double norm = sqrt_normal(c.x * c.x + c.y * c.y);
    const Rcp rn = refined_rcp(norm);
    double2 n = make_double2(div_fast(c.x, rn), div_fast(c.y, rn));
    if (__builtin_expect(!(div_ok(c.x, rn) & div_ok(c.y, rn)), 0)) n = make_double2(div_shared(c.x, rn), div_shared(c.y, rn));
    return dij_of(n, norm, I, J, ovh_i, ovh_j, sql, sqr, K, r16,
                  err);
}

// dlam is compute_dij's value for this entry (from the dt pass or computed inline).
template <bool ALPHA>
__device__ __forceinline__ void first_order_dmu(const double2 c, double v1i, double v2i, double v1j, double v2j,
                                                double dlam, double ai, const double* __restrict__ alpha, int j,
                                                double& d, double& mu) {
    d = dlam;
    mu = mu_of(c.x, c.y, v1i, v2i, v1j, v2j);
    d = fmaxF(d, mu);
    if constexpr (ALPHA) {
        const double s = fmaxF(ai, alpha[j]);
        d = d * s;
        mu = mu * s;
    }
}

// alpha_i from its row sums num = sum(h_j - h_i), denom = sum|h_j - h_i|.
__device__ __forceinline__ double alpha_value(double num, double denom, double hi, double htiny) {
    double a = 1.0;
    if (!(hi <= htiny)) {
        if (!(denom <= fabs(num))) a = fabs(num) / (denom);
        a = a * a;
        a = a * a;
        a = a * a;
    }
    return a;
}

// alpha_limit, first loop (update.f90:758-781) for row i: alpha_i = (|sum(h_j-h_i)| /
// sum|h_j-h_i|)**8, 1 if h_i <= htiny or the denominator does not exceed the numerator.  All index
// loads, then all gathers, then the sums in entry order.
__device__ __forceinline__ double alpha_of(const Mesh& M, const Node* __restrict__ U, int i, double hi, double htiny) {
    double a = 1.0;
    if (!(hi <= htiny)) {
        const int64_t pb = row_base(M, i);
        const int len = M.len[i];
        constexpr int kUnroll = 12;
        int js[kUnroll];
        double hs[kUnroll];
#pragma unroll
        for (int q = 0; q < kUnroll; ++q) js[q] = (q < len) ? (int)M.dcol[pb + 64 * q] : 0;
#pragma unroll
        for (int q = 0; q < kUnroll; ++q) js[q] = (js[q] != kColFar) ? i + js[q] : M.col[pb + 64 * q];
#pragma unroll
        for (int q = 0; q < kUnroll; ++q) hs[q] = U[js[q]].h;
        double num = 0.0, denom = 0.0;
#pragma unroll
        for (int q = 0; q < kUnroll; ++q) {
            if (q < len) {
                num = num + hs[q] - hi;
                denom = denom + fabs(hs[q] - hi);
            }
        }
        for (int q = kUnroll; q < len; ++q) {
            const double hj = U[col_at(M, pb + 64 * (int64_t)q, i)].h;
            num = num + hj - hi;
            denom = denom + fabs(hj - hi);
        }
        a = alpha_value(num, denom, hi, htiny);
    }
    return a;
}

// Per-instance step bookkeeping after the dt pass (SOURCES/main.f90:61-91):
// an instance takes the step while time < tfinal (and its step limit and error flags allow);
// dt = CFL*1/MAXVAL(ABS(d_ii)/m_i); the boundary values of the three stages are evaluated at
// t+dt, (t+dt)+dt/2 and (t+dt/2)+dt; time = to + dt.  advance = 0 only computes dt.  vmax is the pass's
// maximum of the instance (which the caller resets), flags its checks.
__device__ __forceinline__ void finalize_one(InstDev* __restrict__ T, unsigned long long vmax, int flags, int k,
                                             int advance) {
    InstDev& D = T[k];
    if (D.state == INST_FREE) return;
    const double mx = __longlong_as_double((long long)vmax);
    if (!advance) {
        D.dt = D.K.cfl * 1.0 / mx;
        return;
    }
    if (D.state != INST_RUNNING) {
        D.go = 0;
        return;
    }
    if (!takes_steps(D, flags)) {
        D.go = 0;
        D.state = flags ? INST_FAILED : INST_DONE;
        return;
    }
    // test 9 takes the driver's fixed dt and skips COMPUTE_DT (main.f90:66-71)
    const double dt = (D.K.dt_fixed > 0.0) ? D.K.dt_fixed : D.K.cfl * 1.0 / mx;
    const double to = D.time;
    D.dt = dt;
    if (D.bc_kind == SWE_BC_INFLOW) {
        double t = to;
        const double ts0 = t + dt;
        t = to + dt;
        const double ts1 = t + dt / 2;
        t = to + dt / 2;
        const double ts2 = t + dt;
        D.bc_val[0] = D.bc_amp * sin_rn(2.0 * kPi * ts0 / D.bc_period);
        D.bc_val[1] = D.bc_amp * sin_rn(2.0 * kPi * ts1 / D.bc_period);
        D.bc_val[2] = D.bc_amp * sin_rn(2.0 * kPi * ts2 / D.bc_period);
    }
    if (D.dt_log) D.dt_log[D.steps % D.dt_cap] = dt;
    D.time = to + dt;
    D.steps = D.steps + 1;
    D.go = 1;
}

// Antidiffusive flux f_ij of compute_fct_matrix (update.f90:732-745) for an off-diagonal entry,
// with the high-order viscosities MIN(dL, resij), MIN(muL, resij) of update.f90:233-239.
__device__ __forceinline__ double fct_flux(const Node& I, const Node& J, double dLp, double muLp,
                                           double rij, double& dH, double& muH, double& ratij, double& ratji) {
    dH = fminF(dLp, 1.0 * rij);
    muH = fminF(muLp, 1.0 * rij);
    const double zmax = fmaxF(I.z, J.z);
    const double Hij = fmaxF(0.0, I.h + I.z - zmax);
    const double Hji = fmaxF(0.0, J.h + J.z - zmax);
    ratij = (I.h <= 0.0) ? 0.0 : Hij / I.h;
    ratji = (J.h <= 0.0) ? 0.0 : Hji / J.h;
    return (dH - dLp) * (J.h * ratji - I.h * ratij) + (muH - muLp) * (J.h * (1.0 - ratji) - I.h * (1.0 - ratij));
}

// pTilde (update.f90:515-518) at node n: paper_constant = lambdaSGN*g/(3*SQRT(lumped)),
// x = (h*eta)/h**2; the literal integer powers are products from the left, as flang expands them.
__device__ __forceinline__ double sgn_ptilde(double h, double he, double m, const Consts& K) {
    const double pc = K.lambda_sgn * K.g / (3.0 * sqrt_rn(m));
    const double x = he / (h * h);
    return pc * (h * h * h) * (2.0 + 4.0 * (x * x * x) - 6.0 * (x * x * x * x));
}

// bdy (SOURCES/main.f90:176-188) of one row whose Dirichlet components are the bits of mask (1 h, 2 qx, 4 qy):
// the wall and inflow programs, whose values follow from the instance's record.  (Given values come from
// the boundary list: k_bdy.)
__device__ __forceinline__ void bdy_row(Node& o, int mask, const InstDev& D, int stage) {
    const int kind = D.bc_kind;
    if (kind != SWE_BC_WALLS && kind != SWE_BC_INFLOW) return;
    if ((mask & 1) && kind == SWE_BC_INFLOW) o.h = fmaxF(D.bc_level - o.z + D.bc_val[stage], 0.0);
    if (mask & 2) o.qx = 0.0;
    if (mask & 4) o.qy = 0.0;
}

}  // namespace
}  // namespace swe
