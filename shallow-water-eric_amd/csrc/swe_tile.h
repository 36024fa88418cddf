// swe_tile.h -- what the tile kernels (swe_tiles.hip: a lane per row; swe_quads.hip: four lanes per row) share: the
// staged node records and the per-node, per-entry and per-row arithmetic.
#pragma once
#include <hip/hip_runtime.h>

#include "swe_engine.h"
#include "swe_kernels.h"
#include "swe_rows.h"

namespace swe {
namespace {

// MAX(0, h + zb - zb)/h, the depth ratio of a node against its own bed (smb_2: U_i's ratio where its bed is
// the higher one).
__device__ __forceinline__ double own_ratio(double h, double z) { return fmaxF(0.0, h + z - z) / h; }

// The depth ratios of an entry before the dry-node rule: qij = MAX(0, h_i + z_i - zmax)/h_i, qji likewise
// for j, zmax = MAX(z_i, z_j); qi, qj are own_ratio of the two nodes.
__device__ __forceinline__ void depth_ratios(double hi, double zi, double qi, double hj, double zj, double qj,
                                             double& Hij, double& Hji, double& qij, double& qji) {
    const bool up = zi > zj;
    const double zmax = up ? zi : zj;
    Hij = fmaxF(0.0, hi + zi - zmax);
    Hji = fmaxF(0.0, hj + zj - zmax);
    const double quo = (up ? Hji : Hij) / (up ? hj : hi);
    qij = up ? qi : quo;
    qji = up ? quo : qj;
}

// Sums of one row over its entries, for lo_finish.
struct LoSums {
    double r1, r2, r3, fix, e1, e2, e3, emax, emin;
};

// What k_tile_lo stages per node: 80 bytes, read in 16-byte pieces.
struct alignas(16) LoNode {
    double h, z, qx, qy;
    double ovh, sq;       // one_over_h, SQRT(g*ABS(h))
    double q, E;          // own_ratio, entropy
    double alpha, pad;
};

// What k_tile_lo and k_quad_lo do with a row's sums: the low-order solution and the entropy residual.
template <bool WRITE_LO, bool HAS_SRC>
__device__ __forceinline__ void lo_finish(const Node& I, double ovh_i, double E, const LoSums& s, double mi, double dt,
                                          const Consts& K, int roundoff, int i, double* __restrict__ ulo_h,
                                          double2* __restrict__ ulo_q, double* __restrict__ res, int& err) {
    const double v1i = I.qx * ovh_i, v2i = I.qy * ovh_i;
    double e1 = s.e1, e2 = s.e2, e3 = s.e3;
    add_sources<HAS_SRC>(K.src, I, mi, v1i, v2i, dt, K, e2, e3);
    if (WRITE_LO) {
        double r1 = s.r1, r2 = s.r2, r3 = s.r3;
        add_sources<HAS_SRC>(K.src, I, mi, v1i, v2i, dt, K, r2, r3);
        r1 = r1 / mi;
        r2 = r2 / mi;
        r3 = r3 / mi;
        double hL;
        if (roundoff) hL = I.h * (1.0 + dt * s.fix / mi) + dt * r1;
        else hL = fmaxF(I.h + dt * r1, 0.0);
        st_entry1(ulo_h + i, hL);
        st_entry(ulo_q + i, make_double2(I.qx + dt * r2, I.qy + dt * r3));
        if (K.check_h && hL < 0.0) err |= FLAG_NEG_H;
    }
    // entropy_residual (update.f90:838-868)
    e1 = e1 / mi;
    e2 = e2 / mi;
    e3 = e3 / mi;
    const double ht = I.h + dt * e1;
    const double qxt = I.qx + dt * e2;
    const double qyt = I.qy + dt * e3;
    const double ovt = ovh_of(ht, K.htiny);
    const double vn1 = qxt * ovt, vn2 = qyt * ovt;
    double En = K.g * (ht * ht);
    En = En + vn1 * qxt;
    En = En + vn2 * qyt;
    En = 0.5 * En;
    double Ep0 = K.g * I.h;
    Ep0 = Ep0 - 0.5 * (v1i * v1i);
    Ep0 = Ep0 - 0.5 * (v2i * v2i);
    double r = mi * (En - E) / dt;
    r = r - mi * e1 * Ep0;
    r = r - mi * e2 * v1i;
    r = r - mi * e3 * v2i;
    const double rescale = fabs(s.emax - s.emin) / 2.0 + K.ent_cst;
    res[i] = fabs(r) / rescale;
}

template <bool D0>
__device__ __forceinline__ LoNode lo_node(const Node& A, double alpha, const Consts& K) {
    LoNode n;
    n.h = A.h;
    n.z = A.z;
    n.qx = A.qx;
    n.qy = A.qy;
    n.ovh = ovh_of(A.h, K.htiny);
    n.sq = D0 ? 0.0 : sqrt_rn(K.g * fabs(A.h));
    n.q = own_ratio(A.h, A.z);
    // entropy (update.f90:924-935)
    double E = K.g * (A.h * A.h);
    E = E + (A.qx * n.ovh) * A.qx;
    E = E + (A.qy * n.ovh) * A.qy;
    n.E = 0.5 * E;
    n.alpha = alpha;
    return n;
}

// What the limiter passes stage per node.
struct alignas(16) FluxNode {
    double h, z, q, res;   // q: own_ratio
};
struct alignas(16) ApplyNode {
    double h, z, q, res, qx, qy, Rm, pad;
};

// Antidiffusive flux of an off-diagonal entry (fct_flux of swe_rows.h, the depth ratios from the staged nodes).
template <class N>
__device__ __forceinline__ double tile_flux(const N& I, const N& J, const double2 lo, double& dA, double& muA,
                                            double& ratij, double& ratji) {
    const double rij = fmaxF(I.res, J.res);
    dA = fminF(lo.x, 1.0 * rij) - lo.x;
    muA = fminF(lo.y, 1.0 * rij) - lo.y;
    double Hij, Hji;
    depth_ratios(I.h, I.z, I.q, J.h, J.z, J.q, Hij, Hji, ratij, ratji);
    ratij = (I.h <= 0.0) ? 0.0 : ratij;
    ratji = (J.h <= 0.0) ? 0.0 : ratji;
    return dA * (J.h * ratji - I.h * ratij) + muA * (J.h * (1.0 - ratji) - I.h * (1.0 - ratij));
}

struct alignas(16) StageNode {
    double h, z, qx, qy, ovh, sq, q, alpha;
};

// The Euler update of the depth and the RK combination with the walls and inflow of bdy.
template <int SMB>
__device__ __forceinline__ double stage_depth(double h, double dt, double fix, double mi, double r1) {
    if constexpr (SMB == SMB_1) return h + dt * r1;
    else if constexpr (SMB == SMB_ROUNDOFF) return h * (1.0 + dt * fix / mi) + dt * r1;
    else return fmaxF(h + dt * r1, 0.0);
}
__device__ __forceinline__ void stage_out(Node o, const Mesh& M, const InstDev& D, const Node* __restrict__ Uo,
                                          Node* __restrict__ out, int i, int stage, int bdy) {
    if (stage != 0) {
        const Node P = Uo[i];
        o.h = rk_combine(stage, P.h, o.h);
        o.qx = rk_combine(stage, P.qx, o.qx);
        o.qy = rk_combine(stage, P.qy, o.qy);
    }
    if (bdy) {
        const int mask = M.dirm[i];
        if (mask) bdy_row(o, mask, D, stage);
    }
    out[i] = o;
}

struct alignas(16) DtNode {
    double h, qx, qy, ovh, sq, pad;
};

// The end of the dt pass for a workgroup whose lanes hold their rows' values v (>= 0): the maximum and the checks
// of its instance, and with advance, in the workgroup that ends last, finalize_one for every instance.
__device__ __forceinline__ void dt_finish(InstDev* __restrict__ T, double v, int err, int inst,
                                          unsigned long long* __restrict__ vmax, int* __restrict__ flags,
                                          unsigned* __restrict__ done, unsigned long long* red, int* last, int advance,
                                          int ninst) {
    if (err) {
        atomicOr(flags + inst, err);
        __builtin_amdgcn_s_waitcnt(0);    // done before this workgroup's arrival below
    }
    // v >= 0 orders like its bit pattern
    unsigned long long b = (unsigned long long)__double_as_longlong(v);
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(b, off, 64);
        b = (o > b) ? o : b;
    }
    const int tid = (int)threadIdx.x, R = (int)blockDim.x;
    if ((tid & 63) == 0) red[tid >> 6] = b;
    __syncthreads();
    if (tid == 0) {
        unsigned long long mx = 0ull;
        for (int k = 0; k < R / 64; ++k) mx = (red[k] > mx) ? red[k] : mx;
        // most workgroups find a greater maximum already there and leave the word alone
        if (mx > __hip_atomic_load(vmax + inst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(vmax + inst, mx);
    }
    if (!advance) return;
    // The workgroup's flags and maximum are in place before its arrival counts (each thread waits for its own
    // atomics), so the workgroup that arrives last sees all of them; it reads them with atomics, which bypass
    // what its XCD may have cached.
    // Arrivals count in kDoneGroups words first and then, once per word, in one: a single word serialises them
    // (1568 workgroups: 31 us for the pass, 22 us with half as many).
    if (tid == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        const unsigned n = gridDim.x, g = blockIdx.x % kDoneGroups;
        const unsigned groups = n < kDoneGroups ? n : kDoneGroups, members = (n - g + kDoneGroups - 1) / kDoneGroups;
        unsigned* mine = done + kDoneStride * (1 + g);
        int end = 0;
        if (atomicAdd(mine, 1u) == members - 1) {
            atomicExch(mine, 0u);
            if (atomicAdd(done, 1u) == groups - 1) {
                atomicExch(done, 0u);
                end = 1;
            }
        }
        *last = end;
    }
    __syncthreads();
    if (!*last) return;
    for (int k = tid; k < ninst; k += R) {
        const unsigned long long mx = atomicExch(vmax + k, 0ull);
        const int f = __hip_atomic_load(flags + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        finalize_one(T, mx, f, k, 1);
    }
}

}  // namespace
}  // namespace swe
