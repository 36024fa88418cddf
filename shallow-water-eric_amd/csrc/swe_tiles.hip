// swe_tiles.hip -- the step's passes over tiles: one workgroup per tile (up to 4 consecutive slices of an
// instance, swe_layout.h), one lane per row as in swe_kernels.hip, with the node data of the tile's rows and
// of its halo staged in LDS first.
//
// What this changes against the gather kernels: an entry's column is a 16-bit LDS index that streams in
// with c_ij, so no load depends on a loaded index (the gather kernels wait about 1700 cycles for each
// neighbour record); everything that depends on one node only (one_over_h, SQRT(g h), the entropy, the
// depth ratio against the node's own bed) is evaluated once per staged node instead of once per entry, about
// 1.2 instead of 7 times per row; and of the two depth ratios of an entry the one whose bed is the
// higher is that staged quantity, so one division is left of two.  Every expression is the gather kernels',
// on the same operands, so the results are the same bits.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "swe_engine.h"
#include "swe_kernels.h"
#include "swe_tile.h"

namespace swe {

namespace {

// What every kernel reads first.  On a small mesh a kernel's time is the chain of dependent loads (about 0.7 us
// each, nothing being cached across a launch), so all that can be is loaded without waiting for anything
// else: a launch over one instance knows its slices and instance from its arguments, the row's data, the
// halo's rows and the instance's record are loaded side by side, and whether the instance steps at all
// decides afterwards (by emptying the rows) what happens to them.
struct TileHead {
    int s0, nsl;          // first slice and slices of the tile
    int inst;             // its instance
    int tid, w, i;        // thread, wave, global row (of the tile's last slice for waves past it)
    bool own;             // the wave has a slice of the tile
    int len, nhalo;       // entries of the row (0 past the tile), rows of the halo
    int64_t pb;           // first slot of the row
    int64_t hbase;        // start of the halo list
    int hrow;             // this thread's first row of the halo (if it has one)
};
__device__ __forceinline__ TileHead tile_head(const Mesh& M, int remap) {
    TileHead h;
    const int b = remap ? xcd_block() : (int)blockIdx.x;
    const int ts = (int)(blockDim.x >> 6);
    h.tid = (int)threadIdx.x;
    h.w = __builtin_amdgcn_readfirstlane(h.tid >> 6);
    SliceInfo S;
    if (M.one >= 0) {
        h.s0 = M.one_slice0 + b * ts;
        const int left = M.one_nsl - b * ts;
        h.nsl = (left < ts) ? left : ts;
        h.inst = M.one;
        S = M.sl[h.s0];
    } else {
        h.s0 = __builtin_amdgcn_readfirstlane(M.tact[b]);
        S = M.sl[h.s0];
        h.nsl = S.tile_slices;
        h.inst = S.inst;
    }
    h.nhalo = S.nhalo;
    h.own = h.w < h.nsl;
    const int sw = h.own ? h.s0 + h.w : h.s0 + h.nsl - 1;
    h.i = sw * 64 + (h.tid & 63);
    h.len = M.len[h.i];
    h.hbase = (int64_t)h.s0 * kHaloStride;
    h.hrow = M.halo[h.hbase + (h.tid < kHaloStride ? h.tid : kHaloStride - 1)];
    h.pb = M.sl[sw].sbase + (h.tid & 63);
    if (!h.own) h.len = 0;
    return h;
}
// put(k, row) for the nodes of the tile: k = 0..rows-1 its rows (padding rows of its slices too), then its halo.
template <class F>
__device__ __forceinline__ void stage_nodes(const TileHead& h, const Mesh& M, bool go, F&& put) {
    const int R = (int)blockDim.x;
    if (h.own) put(h.tid, h.i);
    if (go) {
        if (h.tid < h.nhalo) put(R + h.tid, h.tid < kHaloStride ? h.hrow : M.halo[h.hbase + h.tid]);
        for (int k = h.tid + R; k < h.nhalo; k += R) put(R + k, M.halo[h.hbase + k]);
    }
}

// Whether a lane writes its entry of the viscosities: each off-diagonal one, and a zero in the diagonal's slot
// (which nothing reads) where most of the wave's lanes are at off-diagonal entries, because a line written
// with holes costs more than a whole one.  1M-node unstructured mesh: k_tile_lo with the dt pass's d_ij 89.0 ->
// 76.9 us, without 107.8 -> 104.9, k_tile_dt 75.1 -> 72.8.  On a lattice, where most lanes meet the diagonal at
// once, that slot stays unwritten: 16.8M nodes, 1378 -> 1393 us against 1411 with the slot always written.
__device__ __forceinline__ bool stores(bool off) {
    if (2 * __popcll(__ballot(off)) >= __popcll(__ballot(true))) return true;
    return off;
}

// The row loop of k_tile_lo (the sums of fct_lo_body in swe_kernels.hip).  WET: every node of the tile and its
// halo is deeper than the dry-node thresholds of both sums, so the ratios need no selection and the two
// sums' momentum parts are one.
template <bool WET, bool ALPHA, bool WRITE_LO, bool D0>
__device__ __forceinline__ void lo_rows(const LoNode* __restrict__ nodes, const Mesh& M, int64_t pb, int len,
                                        const Node& I, const Consts& K, const Rcp& r16, const double* __restrict__ d0,
                                        double2* __restrict__ dmu, int roundoff, LoSums& s, int& err) {
    const int tid = (int)threadIdx.x;
    const double ovh_i = nodes[tid].ovh, sql = nodes[tid].sq, qi = nodes[tid].q;
    const double ai = ALPHA ? nodes[tid].alpha : 1.0;
    const double v1i = I.qx * ovh_i, v2i = I.qy * ovh_i;
    const double thr_lo = roundoff ? K.htiny : 0.0;
    double r1 = 0.0, r2 = 0.0, r3 = 0.0, fix = 0.0, e1 = 0.0, e2 = 0.0, e3 = 0.0, emax = 0.0, emin = 0.0;
    bool split = false;
    double2 c_next = ld_entry(M.c + pb);
    int l_next = M.lcol[pb];
    double d_next = D0 ? ld_entry1(d0 + pb) : 0.0;
    for (int q = 0; q < len; ++q) {
        const int64_t p = pb + 64 * (int64_t)q;
        const double2 c = c_next;
        const int l = l_next;
        const double d0p = d_next;
        if (q + 1 < len) {
            c_next = ld_entry(M.c + p + 64);
            l_next = M.lcol[p + 64];
            if constexpr (D0) d_next = ld_entry1(d0 + p + 64);
        }
        const LoNode& n = nodes[l];
        const Node J{n.h, n.qx, n.qy, n.z};
        const double ovh_j = n.ovh;
        const double v1j = J.qx * ovh_j, v2j = J.qy * ovh_j;
        double Hij, Hji, qij, qji;
        depth_ratios(I.h, I.z, qi, J.h, J.z, n.q, Hij, Hji, qij, qji);
        const double ratij0 = (!WET && I.h <= 0.0) ? 0.0 : qij;
        const double ratji0 = (!WET && J.h <= 0.0) ? 0.0 : qji;
        const double ratijr = (!WET && I.h <= thr_lo) ? 0.0 : qij;
        const double ratjir = (!WET && J.h <= thr_lo) ? 0.0 : qji;
        const bool off = (l != tid);
        double d = 0.0, mu = 0.0;
        if (off) {
            d = D0 ? d0p : dij_from_c(c, I, J, ovh_i, ovh_j, sql, n.sq, K, r16, err);
            mu = mu_of(c.x, c.y, v1i, v2i, v1j, v2j);
            d = fmaxF(d, mu);
            if constexpr (ALPHA) {
                const double a = fmaxF(ai, n.alpha);
                d = d * a;
                mu = mu * a;
            }
        }
        if (stores(off)) st_entry(dmu + p, make_double2(d, mu));
        const double xm = -(c.x * (v1j)) - c.y * (v2j);
        const double xe = -(c.x * (v1j * J.h)) - c.y * (v2j * J.h);
        const double xx2 = -(c.x * (v1j * J.qx)) - c.y * (v2j * J.qx);
        const double xx3 = -(c.x * (v1j * J.qy)) - c.y * (v2j * J.qy);
        const double topo = K.g * I.h * (J.h + J.z - I.h - I.z);
        if (!WET && WRITE_LO && !split && !(ratjir == ratji0 && ratijr == ratij0)) {
            split = true;
            e2 = r2;
            e3 = r3;
        }
        if (WRITE_LO) {
            if (roundoff) {
                if (!off) fix = fix + xm;
                else {
                    fix = fix - mu + (d - mu) * (-ratijr);
                    r1 = r1 + (xm + mu) * J.h + posF((d - mu) * Hji);
                }
            } else {
                r1 = r1 + xe;
                if (off) r1 = r1 + d * (J.h * ratjir - I.h * ratijr) + mu * (J.h * (1.0 - ratjir) - I.h * (1.0 - ratijr));
            }
        }
        // the low-order momentum sums; without them (entropy viscosity alone) the residual's
        r2 = r2 + xx2;
        r3 = r3 + xx3;
        e1 = e1 + xe;
        if (off) {
            const double a = WRITE_LO ? ratjir : ratji0, b = WRITE_LO ? ratijr : ratij0;
            r2 = r2 + d * (J.qx * a - I.qx * b) + mu * (J.qx * (1.0 - a) - I.qx * (1.0 - b));
            r3 = r3 + d * (J.qy * a - I.qy * b) + mu * (J.qy * (1.0 - a) - I.qy * (1.0 - b));
            e1 = e1 + d * (J.h * ratji0 - I.h * ratij0) + mu * (J.h * (1.0 - ratji0) - I.h * (1.0 - ratij0));
        }
        r2 = r2 - topo * c.x;
        r3 = r3 - topo * c.y;
        if (!WET && split) {
            e2 = e2 + xx2;
            e3 = e3 + xx3;
            if (off) {
                e2 = e2 + d * (J.qx * ratji0 - I.qx * ratij0) + mu * (J.qx * (1.0 - ratji0) - I.qx * (1.0 - ratij0));
                e3 = e3 + d * (J.qy * ratji0 - I.qy * ratij0) + mu * (J.qy * (1.0 - ratji0) - I.qy * (1.0 - ratij0));
            }
            e2 = e2 - topo * c.x;
            e3 = e3 - topo * c.y;
        }
        const double Ej = n.E;
        if (q == 0) {
            emax = Ej;
            emin = Ej;
        } else {
            emax = (Ej > emax) ? Ej : emax;
            emin = (Ej < emin) ? Ej : emin;
        }
    }
    if (!split) {
        e2 = r2;
        e3 = r3;
    }
    s = LoSums{r1, r2, r3, fix, e1, e2, e3, emax, emin};
}

// =============================================================================================
// FCT / entropy-viscosity stage, pass 1 on tiles: k_fct_lo's results (viscosities dmu, low-order solution,
// entropy residual).
// =============================================================================================
template <bool ALPHA, bool WRITE_LO, bool HAS_SRC, bool D0>
__global__ void __launch_bounds__(64 * kMaxTileSlices, 4)
k_tile_lo(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, double* __restrict__ ulo_h,
          double2* __restrict__ ulo_q, double2* __restrict__ dmu, double* __restrict__ res,
          const double* __restrict__ d0, const double* __restrict__ alpha, int roundoff, int* __restrict__ flags_out,
          int remap) {
    extern __shared__ double smem[];
    LoNode* nodes = (LoNode*)smem;
    const TileHead h = tile_head(M, remap);
    const int inst = h.inst, tid = h.tid, i = h.i;
    const bool go = T[inst].go != 0;
    const Consts K = T[inst].K;
    const double dt = T[inst].dt;
    const int len = go ? h.len : 0;
    const double wet_h = fmaxF(K.htiny, 0.0);
    bool wet = true;
    auto put = [&](int k, int row) {
        const Node A = U[row];
        const LoNode n = lo_node<D0>(A, ALPHA ? alpha[row] : 0.0, K);
        nodes[k] = n;
        // (padding rows of the tile's slices, which nothing refers to, do not count)
        wet = wet && (A.h > wet_h || (k == tid && len == 0));
    };
    stage_nodes(h, M, go, put);
    const bool all_wet = __syncthreads_and(wet ? 1 : 0) != 0;
    if (len == 0) return;
    const Rcp r16 = uniform_rcp(K.g16);
    const Node I{nodes[tid].h, nodes[tid].qx, nodes[tid].qy, nodes[tid].z};
    int err = 0;
    LoSums s;
    if (all_wet) lo_rows<true, ALPHA, WRITE_LO, D0>(nodes, M, h.pb, len, I, K, r16, d0, dmu, roundoff, s, err);
    else lo_rows<false, ALPHA, WRITE_LO, D0>(nodes, M, h.pb, len, I, K, r16, d0, dmu, roundoff, s, err);
    lo_finish<WRITE_LO, HAS_SRC>(I, nodes[tid].ovh, nodes[tid].E, s, M.m[i], dt, K, roundoff, i, ulo_h, ulo_q, res, err);
    raise_flag(flags_out, inst, err);
}

// =============================================================================================
// FCT stage, pass 2 on tiles: k_fct_rminus's R-.
// =============================================================================================
// Entries a lane holds in registers: their viscosities and columns are loaded before the staging barrier, all
// at once; longer rows read the rest in a loop.
constexpr int kHeld = 8;

struct HeldRow {
    double2 lo[kHeld];
    int l[kHeld];
};
__device__ __forceinline__ void hold_row(HeldRow& H, const Mesh& M, const double2* __restrict__ dmu, int64_t pb, int len) {
#pragma unroll
    for (int q = 0; q < kHeld; ++q)
        if (q < len) {
            H.lo[q] = ld_entry(dmu + pb + 64 * q);
            H.l[q] = M.lcol[pb + 64 * q];
        }
}

__global__ void __launch_bounds__(64 * kMaxTileSlices)
k_tile_rminus(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, const double* __restrict__ ulo_h,
              const double2* __restrict__ dmu, const double* __restrict__ res, double* __restrict__ Rm, int remap) {
    extern __shared__ double smem[];
    FluxNode* nodes = (FluxNode*)smem;
    const TileHead h = tile_head(M, remap);
    const int inst = h.inst, tid = h.tid, i = h.i;
    const bool go = T[inst].go != 0;
    const double dt = T[inst].dt;
    const double htiny = T[inst].K.htiny;
    const int len = go ? h.len : 0;
    const int64_t pb = h.pb;
    HeldRow H;
    hold_row(H, M, dmu, pb, len);
    auto stage = [&](int k, int row) {
        const Node A = U[row];
        nodes[k] = FluxNode{A.h, A.z, own_ratio(A.h, A.z), res[row]};
    };
    stage_nodes(h, M, go, stage);
    __syncthreads();
    if (len == 0) return;
    const FluxNode I = nodes[tid];
    double P = -1.0e-15;
    auto entry = [&](const double2 lo, int l) {
        if (l == tid) return;    // f_ii is a zero, never < 0
        double dA, muA, rij_, rji_;
        const double f = tile_flux(I, nodes[l], lo, dA, muA, rij_, rji_);
        if (f < 0.0) P = P + f;
    };
#pragma unroll
    for (int q = 0; q < kHeld; ++q)
        if (q < len) entry(H.lo[q], H.l[q]);
    for (int q = kHeld; q < len; ++q) entry(ld_entry(dmu + pb + 64 * q), M.lcol[pb + 64 * q]);
    const double scaled = (M.m[i] / dt) * ulo_h[i];
    const double Q = 0.0 - scaled;
    double Ri = fminF(Q / P, 1.0);
    if (scaled <= htiny) Ri = 0.0;
    Rm[i] = Ri;
}

// =============================================================================================
// FCT stage, pass 3 on tiles: k_fct_apply's limited update and RK combination, with the wall and inflow
// values of bdy.
// =============================================================================================
__global__ void __launch_bounds__(64 * kMaxTileSlices)
k_tile_apply(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, const Node* __restrict__ Uo,
             const double* __restrict__ ulo_h, const double2* __restrict__ ulo_q, Node* __restrict__ out,
             const double2* __restrict__ dmu, const double* __restrict__ res, const double* __restrict__ Rm, int stage,
             int bdy, int* __restrict__ flags_out, int remap) {
    extern __shared__ double smem[];
    ApplyNode* nodes = (ApplyNode*)smem;
    const TileHead h = tile_head(M, remap);
    const int inst = h.inst, tid = h.tid, i = h.i;
    const bool go = T[inst].go != 0;
    const double dt = T[inst].dt;
    const int check_h = T[inst].K.check_h;
    const int len = go ? h.len : 0;
    const int64_t pb = h.pb;
    HeldRow H;
    hold_row(H, M, dmu, pb, len);
    auto put = [&](int k, int row) {
        const Node A = U[row];
        nodes[k] = ApplyNode{A.h, A.z, own_ratio(A.h, A.z), res[row], A.qx, A.qy, Rm[row], 0.0};
    };
    stage_nodes(h, M, go, put);
    __syncthreads();
    if (len == 0) return;
    const ApplyNode I = nodes[tid];
    double x1 = 0.0, x2 = 0.0, x3 = 0.0;
    auto entry = [&](const double2 lo, int l) {
        if (l == tid) return;    // contributes d*(0) + mu*(0)
        const ApplyNode& J = nodes[l];
        double dA, muA, ratij, ratji;
        const double f = tile_flux(I, J, lo, dA, muA, ratij, ratji);
        const double lim = (f >= 0.0) ? J.Rm : I.Rm;
        const double d = dA * lim;
        const double mu = muA * lim;
        const double a = 1.0 - ratji, b = 1.0 - ratij;
        x1 = x1 + d * (J.h * ratji - I.h * ratij) + mu * (J.h * a - I.h * b);
        x2 = x2 + d * (J.qx * ratji - I.qx * ratij) + mu * (J.qx * a - I.qx * b);
        x3 = x3 + d * (J.qy * ratji - I.qy * ratij) + mu * (J.qy * a - I.qy * b);
    };
#pragma unroll
    for (int q = 0; q < kHeld; ++q)
        if (q < len) entry(H.lo[q], H.l[q]);
    for (int q = kHeld; q < len; ++q) entry(ld_entry(dmu + pb + 64 * q), M.lcol[pb + 64 * q]);
    const double mi = M.m[i];
    const double hL = ld_entry1(ulo_h + i);   // low-order solution of k_tile_lo
    const double2 qL = ld_entry(ulo_q + i);
    Node o;
    o.h = hL + dt * (x1 / mi);
    o.qx = qL.x + dt * (x2 / mi);
    o.qy = qL.y + dt * (x3 / mi);
    const int err = (check_h && o.h < 0.0) ? FLAG_NEG_H : 0;
    if (stage != 0) {
        const Node P = Uo[i];
        o.h = rk_combine(stage, P.h, o.h);
        o.qx = rk_combine(stage, P.qx, o.qx);
        o.qy = rk_combine(stage, P.qy, o.qy);
    }
    o.z = I.z;
    if (bdy) {
        const int mask = M.dirm[i];
        if (mask) bdy_row(o, mask, T[inst], stage);
    }
    out[i] = o;
    raise_flag(flags_out, inst, err);
}

// =============================================================================================
// First-order stage on tiles: k_stage_lo's update, with the wall and inflow values of bdy.
// =============================================================================================
// Low-order sums of an entry with the neighbour's components uj over the own ui (k_stage_lo's and
// k_stage_sgn's; v2fi, v2fj are the second velocities of the flux).
template <int SMB, int NC>
__device__ __forceinline__ void stage_entry(double (&r)[NC], double& fix, const double (&ui)[NC], const double (&uj)[NC],
                                            double zi, double zj, const double2 c, double v1i, double v2fi, double v1j,
                                            double v2fj, double Hij, double Hji, double ratij, double ratji, double d,
                                            double mu, bool off, const Consts& K) {
    if constexpr (SMB == SMB_1) {
        // smb_1 (update.f90:378-409)
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const double xx = -(c.x * (v1j * uj[k] * ratji + v1i * ui[k] * ratij)) -
                              c.y * (v2fj * uj[k] * ratji + v2fi * ui[k] * ratij);
            r[k] = r[k] + xx;
            if (off) r[k] = r[k] + d * (uj[k] * ratji - ui[k] * ratij);
        }
        if (off) {
            const double t = 0.5 * K.g * (Hji * Hji - Hij * Hij);
            r[1] = r[1] - t * c.x;
            r[2] = r[2] - t * c.y;
        }
    } else {
        constexpr int k0 = (SMB == SMB_ROUNDOFF) ? 1 : 0;
        if constexpr (SMB == SMB_ROUNDOFF) {
            // smb_2_roundoff (update.f90:566-611): mass equation with fix_roundoff
            const double xm = -(c.x * (v1j)) - c.y * (v2fj);
            if (!off) {
                fix = fix + xm;
            } else {
                fix = fix - mu + (d - mu) * (-ratij);
                r[0] = r[0] + (xm + mu) * uj[0] + posF((d - mu) * Hji);
            }
        }
        const double aj = 1.0 - ratji, ai = 1.0 - ratij;
#pragma unroll
        for (int k = k0; k < NC; ++k) {
            // smb_2 (update.f90:656-663)
            const double xx = -(c.x * (v1j * uj[k])) - c.y * (v2fj * uj[k]);
            r[k] = r[k] + xx;
            if (SMB != SMB_GALERKIN && off)
                r[k] = r[k] + d * (uj[k] * ratji - ui[k] * ratij) + mu * (uj[k] * aj - ui[k] * ai);
        }
        const double topo = K.g * ui[0] * (uj[0] + zj - ui[0] - zi);
        r[1] = r[1] - topo * c.x;
        r[2] = r[2] - topo * c.y;
    }
}

template <int SMB, bool ALPHA, bool HAS_SRC, bool D0>
__global__ void __launch_bounds__(64 * kMaxTileSlices)
k_tile_stage(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, const Node* __restrict__ Uo,
             Node* __restrict__ out, const double* __restrict__ d0, const double* __restrict__ alpha, int stage, int bdy,
             int* __restrict__ flags_out, int remap) {
    constexpr bool VISC = SMB != SMB_GALERKIN;
    extern __shared__ double smem[];
    StageNode* nodes = (StageNode*)smem;
    const TileHead h = tile_head(M, remap);
    const int inst = h.inst, tid = h.tid, i = h.i;
    const bool go = T[inst].go != 0;
    const Consts K = T[inst].K;
    const double dt = T[inst].dt;
    const int len = go ? h.len : 0;
    const int64_t pb = h.pb;
    double2 c_next{};
    int l_next = 0;
    double d_next = 0.0;
    if (len > 0) {
        c_next = ld_entry(M.c + pb);
        l_next = M.lcol[pb];
        if constexpr (VISC && D0) d_next = ld_entry1(d0 + pb);
    }
    auto put = [&](int k, int row) {
        const Node A = U[row];
        nodes[k] = StageNode{A.h, A.z, A.qx, A.qy, ovh_of(A.h, K.htiny),
                             (VISC && !D0) ? sqrt_rn(K.g * fabs(A.h)) : 0.0, own_ratio(A.h, A.z),
                             ALPHA ? alpha[row] : 0.0};
    };
    stage_nodes(h, M, go, put);
    __syncthreads();
    if (len == 0) return;
    const Rcp r16 = uniform_rcp(K.g16);
    const StageNode A = nodes[tid];
    const Node I{A.h, A.qx, A.qy, A.z};
    const double v1i = I.qx * A.ovh, v2i = I.qy * A.ovh;
    const double thr = (SMB == SMB_ROUNDOFF || SMB == SMB_1) ? K.htiny : 0.0;
    const double ui[3] = {I.h, I.qx, I.qy};
    double r[3] = {0.0, 0.0, 0.0}, fix = 0.0;
    int err = 0;
    for (int q = 0; q < len; ++q) {
        const int64_t p = pb + 64 * (int64_t)q;
        const double2 c = c_next;
        const int l = l_next;
        const double d0p = d_next;
        if (q + 1 < len) {
            c_next = ld_entry(M.c + p + 64);
            l_next = M.lcol[p + 64];
            if constexpr (VISC && D0) d_next = ld_entry1(d0 + p + 64);
        }
        const StageNode& B = nodes[l];
        const Node J{B.h, B.qx, B.qy, B.z};
        const double v1j = J.qx * B.ovh, v2j = J.qy * B.ovh;
        double Hij, Hji, ratij, ratji;
        depth_ratios(I.h, I.z, A.q, J.h, J.z, B.q, Hij, Hji, ratij, ratji);
        ratij = (I.h <= thr) ? 0.0 : ratij;
        ratji = (J.h <= thr) ? 0.0 : ratji;
        const bool off = (l != tid);
        double d = 0.0, mu = 0.0;
        if (VISC && off) {
            d = D0 ? d0p : dij_from_c(c, I, J, A.ovh, B.ovh, A.sq, B.sq, K, r16, err);
            mu = mu_of(c.x, c.y, v1i, v2i, v1j, v2j);
            d = fmaxF(d, mu);
            if constexpr (ALPHA) {
                const double a = fmaxF(A.alpha, B.alpha);
                d = d * a;
                mu = mu * a;
            }
        }
        const double uj[3] = {J.h, J.qx, J.qy};
        stage_entry<SMB, 3>(r, fix, ui, uj, I.z, J.z, c, v1i, v2i, v1j, v2j, Hij, Hji, ratij, ratji, d, mu, off, K);
    }
    const double mi = M.m[i];
    add_sources<HAS_SRC>(K.src, I, mi, v1i, v2i, dt, K, r[1], r[2]);
    for (int k = 0; k < 3; ++k) r[k] = r[k] / mi;
    const Node o{stage_depth<SMB>(I.h, dt, fix, mi, r[0]), I.qx + dt * r[1], I.qy + dt * r[2], I.z};
    stage_out(o, M, T[inst], Uo, out, i, stage, bdy);
    raise_flag(flags_out, inst, err);
}

// =============================================================================================
// SGN stage on tiles: k_stage_sgn's update.  pTilde (two divisions and a square root) is one of the staged
// terms, once per node.
// =============================================================================================
struct alignas(16) SgnNode {
    double h, z, qx, qy, ovh, sq, q, alpha, he, hw, pt, pad;
};

template <int SMB, bool ALPHA, bool D0>
__global__ void __launch_bounds__(64 * kMaxTileSlices)
k_tile_sgn(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, const NodeX* __restrict__ UX,
           const Node* __restrict__ Uo, const NodeX* __restrict__ UoX, Node* __restrict__ out, NodeX* __restrict__ outX,
           const double* __restrict__ d0, const double* __restrict__ alpha, int stage, int bdy,
           int* __restrict__ flags_out, int remap) {
    constexpr bool VISC = SMB != SMB_GALERKIN;
    extern __shared__ double smem[];
    SgnNode* nodes = (SgnNode*)smem;
    const TileHead h = tile_head(M, remap);
    const int inst = h.inst, tid = h.tid, i = h.i;
    const bool go = T[inst].go != 0;
    const Consts K = T[inst].K;
    const double dt = T[inst].dt;
    const int len = go ? h.len : 0;
    const int64_t pb = h.pb;
    double2 c_next{};
    int l_next = 0;
    double d_next = 0.0;
    if (len > 0) {
        c_next = M.c[pb];
        l_next = M.lcol[pb];
        if constexpr (VISC && D0) d_next = ld_entry1(d0 + pb);
    }
    auto put = [&](int k, int row) {
        const Node A = U[row];
        const NodeX X = UX[row];
        nodes[k] = SgnNode{A.h, A.z, A.qx, A.qy, ovh_of(A.h, K.htiny),
                           (VISC && !D0) ? sqrt_rn(K.g * fabs(A.h)) : 0.0, own_ratio(A.h, A.z),
                           ALPHA ? alpha[row] : 0.0, X.he, X.hw, sgn_ptilde(A.h, X.he, M.m[row], K), 0.0};
    };
    stage_nodes(h, M, go, put);
    __syncthreads();
    if (len == 0) return;
    const Rcp r16 = uniform_rcp(K.g16);
    const SgnNode& A = nodes[tid];
    const Node I{A.h, A.qx, A.qy, A.z};
    const double ovh_i = A.ovh, sql = A.sq, qi = A.q, ai = A.alpha;
    const double v1i = I.qx * ovh_i, v2i = I.qy * ovh_i;
    const double v2fi = I.qy * ovh_i * 0.0;   // velocity(2,i) of the model's flux
    const double thr = (SMB == SMB_ROUNDOFF || SMB == SMB_1) ? K.htiny : 0.0;
    const double ui[5] = {I.h, I.qx, I.qy, A.he, A.hw};
    double r[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, fix = 0.0;
    int err = 0;
    for (int q = 0; q < len; ++q) {
        const int64_t p = pb + 64 * (int64_t)q;
        const double2 c = c_next;
        const int l = l_next;
        const double d0p = d_next;
        if (q + 1 < len) {
            c_next = M.c[p + 64];
            l_next = M.lcol[p + 64];
            if constexpr (VISC && D0) d_next = ld_entry1(d0 + p + 64);
        }
        const SgnNode& B = nodes[l];
        const Node J{B.h, B.qx, B.qy, B.z};
        const double v1j = J.qx * B.ovh, v2j = J.qy * B.ovh;
        const double v2fj = J.qy * B.ovh * 0.0;
        double Hij, Hji, ratij, ratji;
        depth_ratios(I.h, I.z, qi, J.h, J.z, B.q, Hij, Hji, ratij, ratji);
        ratij = (I.h <= thr) ? 0.0 : ratij;
        ratji = (J.h <= thr) ? 0.0 : ratji;
        const bool off = (l != tid);
        double d = 0.0, mu = 0.0;
        if (VISC && off) {
            d = D0 ? d0p : dij_from_c(c, I, J, ovh_i, B.ovh, sql, B.sq, K, r16, err);
            mu = mu_of(c.x, c.y, v1i, v2i, v1j, v2j);
            d = fmaxF(d, mu);
            if constexpr (ALPHA) {
                const double a = fmaxF(ai, B.alpha);
                d = d * a;
                mu = mu * a;
            }
        }
        const double uj[5] = {J.h, J.qx, J.qy, B.he, B.hw};
        stage_entry<SMB, 5>(r, fix, ui, uj, I.z, J.z, c, v1i, v2fi, v1j, v2fj, Hij, Hji, ratij, ratji, d, mu, off, K);
    }
    // mSGN_RHS: the momenta lose pTilde(j)*c_ij over the row in CSR order, then the h*eta and h*w sources
    for (int q = 0; q < len; ++q) {
        const double2 c = M.c[pb + 64 * (int64_t)q];
        const double pt = nodes[M.lcol[pb + 64 * (int64_t)q]].pt;
        r[1] = r[1] - pt * c.x;
        r[2] = r[2] - pt * c.y;
    }
    const double mi = M.m[i];
    {
        const double pc = K.lambda_sgn * K.g / (3.0 * sqrt_rn(mi));
        const double x = ui[3] / (I.h * I.h);
        const double psi = 12.0 * (x - 1.0);
        const double t = ui[3] / I.h;
        const double s = 3.0 * pc * (t * t) * psi;
        r[3] = r[3] + mi * ui[4];
        r[4] = r[4] - mi * s;
    }
    for (int k = 0; k < 5; ++k) r[k] = r[k] / mi;
    const Node o{stage_depth<SMB>(I.h, dt, fix, mi, r[0]), I.qx + dt * r[1], I.qy + dt * r[2], I.z};
    NodeX x{ui[3] + dt * r[3], ui[4] + dt * r[4]};
    if (stage != 0) {
        const NodeX PX = UoX[i];
        x.he = rk_combine(stage, PX.he, x.he);
        x.hw = rk_combine(stage, PX.hw, x.hw);
    }
    outX[i] = x;
    stage_out(o, M, T[inst], Uo, out, i, stage, bdy);
    raise_flag(flags_out, inst, err);
}

// =============================================================================================
// Entropy-viscosity-only stage, pass 2 on tiles: k_ev_update's update.
// =============================================================================================
template <bool HAS_SRC>
__global__ void __launch_bounds__(64 * kMaxTileSlices)
k_tile_ev(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, const Node* __restrict__ Uo,
          Node* __restrict__ out, const double2* __restrict__ dmu, const double* __restrict__ res, int roundoff,
          int stage, int bdy, int* __restrict__ flags_out, int remap) {
    extern __shared__ double smem[];
    StageNode* nodes = (StageNode*)smem;     // alpha holds the residual, sq is unused
    const TileHead h = tile_head(M, remap);
    const int inst = h.inst, tid = h.tid, i = h.i;
    const bool go = T[inst].go != 0;
    const Consts K = T[inst].K;
    const double dt = T[inst].dt;
    const int len = go ? h.len : 0;
    const int64_t pb = h.pb;
    double2 c_next{}, lo_next{};
    int l_next = 0;
    if (len > 0) {
        c_next = ld_entry(M.c + pb);
        lo_next = ld_entry(dmu + pb);
        l_next = M.lcol[pb];
    }
    auto put = [&](int k, int row) {
        const Node A = U[row];
        nodes[k] = StageNode{A.h, A.z, A.qx, A.qy, ovh_of(A.h, K.htiny), 0.0, own_ratio(A.h, A.z), res[row]};
    };
    stage_nodes(h, M, go, put);
    __syncthreads();
    if (len == 0) return;
    const StageNode A = nodes[tid];
    const Node I{A.h, A.qx, A.qy, A.z};
    const double v1i = I.qx * A.ovh, v2i = I.qy * A.ovh;
    const double thr = roundoff ? K.htiny : 0.0;
    const double ui[3] = {I.h, I.qx, I.qy};
    double r[3] = {0.0, 0.0, 0.0}, fix = 0.0;
    for (int q = 0; q < len; ++q) {
        const int64_t p = pb + 64 * (int64_t)q;
        const double2 c = c_next, lo = lo_next;
        const int l = l_next;
        if (q + 1 < len) {
            c_next = ld_entry(M.c + p + 64);
            lo_next = ld_entry(dmu + p + 64);
            l_next = M.lcol[p + 64];
        }
        const StageNode& B = nodes[l];
        const Node J{B.h, B.qx, B.qy, B.z};
        const double v1j = J.qx * B.ovh, v2j = J.qy * B.ovh;
        double Hij, Hji, ratij, ratji;
        depth_ratios(I.h, I.z, A.q, J.h, J.z, B.q, Hij, Hji, ratij, ratji);
        ratij = (I.h <= thr) ? 0.0 : ratij;
        ratji = (J.h <= thr) ? 0.0 : ratji;
        const bool off = (l != tid);
        double d = 0.0, mu = 0.0;
        if (off) {
            const double rij = fmaxF(A.alpha, B.alpha);
            d = fminF(lo.x, 1.0 * rij);
            mu = fminF(lo.y, 1.0 * rij);
        }
        const double uj[3] = {J.h, J.qx, J.qy};
        if (roundoff)
            stage_entry<SMB_ROUNDOFF, 3>(r, fix, ui, uj, I.z, J.z, c, v1i, v2i, v1j, v2j, Hij, Hji, ratij, ratji, d, mu,
                                         off, K);
        else
            stage_entry<SMB_2, 3>(r, fix, ui, uj, I.z, J.z, c, v1i, v2i, v1j, v2j, Hij, Hji, ratij, ratji, d, mu, off, K);
    }
    const double mi = M.m[i];
    add_sources<HAS_SRC>(K.src, I, mi, v1i, v2i, dt, K, r[1], r[2]);
    for (int k = 0; k < 3; ++k) r[k] = r[k] / mi;
    const Node o{roundoff ? stage_depth<SMB_ROUNDOFF>(I.h, dt, fix, mi, r[0]) : stage_depth<SMB_2>(I.h, dt, fix, mi, r[0]),
                 I.qx + dt * r[1], I.qy + dt * r[2], I.z};
    const int err = (K.check_h && o.h < 0.0) ? FLAG_NEG_H : 0;
    stage_out(o, M, T[inst], Uo, out, i, stage, bdy);
    raise_flag(flags_out, inst, err);
}

// =============================================================================================
// alpha_limit's factors on tiles: k_alpha's (the first stage's come from the dt pass).  Bound by latency: the
// columns are loaded while the depths are staged, and no load depends on another but the halo's.  Measured
// against k_alpha: 22.0 -> 12.9 us at 1M nodes, 267 -> 187 at 16.8M, 5.0 -> 4.8 at 100k.
// =============================================================================================
__global__ void __launch_bounds__(64 * kMaxTileSlices)
k_tile_alpha(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, double* __restrict__ alpha, int remap) {
    extern __shared__ double depth[];
    const TileHead h = tile_head(M, remap);
    const int inst = h.inst, tid = h.tid;
    const bool go = T[inst].go != 0;
    const double htiny = T[inst].K.htiny;
    const int len = go ? h.len : 0;
    int l[kHeld];
#pragma unroll
    for (int q = 0; q < kHeld; ++q) l[q] = (q < len) ? (int)M.lcol[h.pb + 64 * q] : tid;
    auto put = [&](int k, int row) { depth[k] = U[row].h; };
    stage_nodes(h, M, go, put);
    __syncthreads();
    if (len == 0) return;
    const double hi = depth[tid];
    double num = 0.0, den = 0.0;
    auto entry = [&](int x) {
        const double hj = depth[x];
        num = num + hj - hi;
        den = den + fabs(hj - hi);
    };
#pragma unroll
    for (int q = 0; q < kHeld; ++q)
        if (q < len) entry(l[q]);
    for (int q = kHeld; q < len; ++q) entry(M.lcol[h.pb + 64 * q]);
    alpha[h.i] = alpha_value(num, den, hi, htiny);
}

// =============================================================================================
// COMPUTE_DT on tiles: k_compute_dt's d_ij (kept in d0 for the first stage) and per-instance maxima, and where
// asked for the first stage's alpha (its neighbours' depths are staged here anyway); with
// advance, the workgroup that ends last does the step's bookkeeping (k_finalize_dt) as well.
// =============================================================================================
__global__ void __launch_bounds__(64 * kMaxTileSlices)
k_tile_dt(Mesh M, InstDev* __restrict__ T, const Node* __restrict__ U, double* __restrict__ d0,
          double* __restrict__ alpha, unsigned long long* __restrict__ vmax, int* __restrict__ flags,
          unsigned* __restrict__ done, int all, int advance, int ninst, int remap) {
    extern __shared__ double smem[];
    DtNode* nodes = (DtNode*)smem;
    __shared__ unsigned long long red[kMaxTileSlices];
    __shared__ int last;
    const TileHead h = tile_head(M, remap);
    const int inst = h.inst, tid = h.tid, i = h.i;
    // (per wave: a check raised meanwhile may end some waves' part; every barrier is met by all of them)
    const bool live = all ? T[inst].state != INST_FREE : takes_steps(T[inst], flags[inst]);
    const int len = live ? h.len : 0;
    const int64_t pb = h.pb;
    const Consts K = T[inst].K;
    double2 c_next{};
    int l_next = 0;
    if (len > 0) {
        c_next = ld_entry(M.c + pb);
        l_next = M.lcol[pb];
    }
    auto put = [&](int k, int row) {
        const Node A = U[row];
        nodes[k] = DtNode{A.h, A.qx, A.qy, ovh_of(A.h, K.htiny), sqrt_rn(K.g * fabs(A.h)), 0.0};
    };
    stage_nodes(h, M, live, put);
    __syncthreads();
    double v = 0.0;
    int err = 0;
    if (len > 0) {
        const Rcp r16 = uniform_rcp(K.g16);
        const DtNode A = nodes[tid];
        const Node I{A.h, A.qx, A.qy, 0.0};
        double s = 0.0, num = 0.0, den = 0.0;
        for (int q = 0; q < len; ++q) {
            const int64_t p = pb + 64 * (int64_t)q;
            const double2 c = c_next;
            const int l = l_next;
            if (q + 1 < len) {
                c_next = ld_entry(M.c + p + 64);
                l_next = M.lcol[p + 64];
            }
            const DtNode& B = nodes[l];
            num = num + B.h - A.h;
            den = den + fabs(B.h - A.h);
            const bool off = (l != tid);
            double d = 0.0;            // the reference's row sum adds a 0.0 there
            if (off) {
                const Node J{B.h, B.qx, B.qy, 0.0};
                d = dij_from_c(c, I, J, A.ovh, B.ovh, A.sq, B.sq, K, r16, err);
                s = s + d;
            }
            if (d0 && stores(off)) st_entry1(d0 + p, d);
        }
        v = fabs(-s) / M.m[i];
        if (alpha) alpha[i] = alpha_value(num, den, A.h, K.htiny);
    }
    dt_finish(T, v, err, inst, vmax, flags, done, red, &last, advance, ninst);
}

template <bool ALPHA, bool WRITE_LO, bool HAS_SRC, bool D0>
void go_tile_lo(Pool& P, const Node* U, const double* d0) {
    const Mesh M = mesh_view(P);
    hipLaunchKernelGGL((k_tile_lo<ALPHA, WRITE_LO, HAS_SRC, D0>), dim3((unsigned)P.ntile), dim3(64 * P.tile_slices),
                       sizeof(LoNode) * (size_t)P.tile_nodes, P.stream, M, (const InstDev*)P.tab, U, P.ulo_h, P.ulo_q,
                       P.dmu, P.res, d0, (const double*)P.alpha, P.mode.roundoff, P.flags, P.tune.k[KID_FCT_LO].remap);
}

template <bool ALPHA, bool WRITE_LO>
void go_tile_lo(Pool& P, const Node* U, const double* d0) {
    if (P.any_src) {
        if (d0) go_tile_lo<ALPHA, WRITE_LO, true, true>(P, U, d0);
        else go_tile_lo<ALPHA, WRITE_LO, true, false>(P, U, d0);
    } else {
        if (d0) go_tile_lo<ALPHA, WRITE_LO, false, true>(P, U, d0);
        else go_tile_lo<ALPHA, WRITE_LO, false, false>(P, U, d0);
    }
}

template <int SMB, bool ALPHA>
void go_tile_stage(Pool& P, const Node* U, const Node* Uo, Node* out, const double* d0, int stage, bool bdy) {
    auto go = [&](auto src, auto has_d0) {
        constexpr bool S = decltype(src)::value, D = decltype(has_d0)::value;
        hipLaunchKernelGGL((k_tile_stage<SMB, ALPHA, S, D>), dim3((unsigned)P.ntile), dim3(64 * P.tile_slices),
                           sizeof(StageNode) * (size_t)P.tile_nodes, P.stream, mesh_view(P), (const InstDev*)P.tab, U,
                           Uo, out, d0, (const double*)P.alpha, stage, bdy ? 1 : 0, P.flags,
                           P.tune.k[KID_STAGE_LO].remap);
    };
    using T_ = std::true_type;
    using F_ = std::false_type;
    constexpr bool visc = SMB != SMB_GALERKIN;
    if (P.any_src) {
        if (visc && d0) go(T_{}, std::bool_constant<visc>{});
        else go(T_{}, F_{});
    } else {
        if (visc && d0) go(F_{}, std::bool_constant<visc>{});
        else go(F_{}, F_{});
    }
}

template <int SMB, bool ALPHA>
void go_tile_sgn(Pool& P, const Node* U, const Node* Uo, Node* out, const double* d0, int stage, bool bdy) {
    auto go = [&](auto has_d0) {
        constexpr bool D = decltype(has_d0)::value;
        hipLaunchKernelGGL((k_tile_sgn<SMB, ALPHA, D>), dim3((unsigned)P.ntile), dim3(64 * P.tile_slices),
                           sizeof(SgnNode) * (size_t)P.tile_nodes, P.stream, mesh_view(P), (const InstDev*)P.tab, U,
                           (const NodeX*)ext_of(P, U), Uo, (const NodeX*)ext_of(P, Uo), out, ext_of(P, out), d0,
                           (const double*)P.alpha, stage, bdy ? 1 : 0, P.flags, P.tune.k[KID_STAGE_LO].remap);
    };
    constexpr bool visc = SMB != SMB_GALERKIN;
    if (visc && d0) go(std::bool_constant<visc>{});
    else go(std::false_type{});
}

template <int SMB>
void go_tile_first(Pool& P, const Node* U, const Node* Uo, Node* out, const double* d0, bool alpha, int stage, bool bdy) {
    if (P.mode.sgn) {
        if (alpha) go_tile_sgn<SMB, SMB != SMB_GALERKIN>(P, U, Uo, out, d0, stage, bdy);
        else go_tile_sgn<SMB, false>(P, U, Uo, out, d0, stage, bdy);
    } else {
        if (alpha) go_tile_stage<SMB, SMB != SMB_GALERKIN>(P, U, Uo, out, d0, stage, bdy);
        else go_tile_stage<SMB, false>(P, U, Uo, out, d0, stage, bdy);
    }
}

}  // namespace

void launch_tile_lo(Pool& P, const Node* U, const double* d0, bool alpha, bool write_lo) {
    if (write_lo) {
        if (alpha) go_tile_lo<true, true>(P, U, d0);
        else go_tile_lo<false, true>(P, U, d0);
    } else {
        if (alpha) go_tile_lo<true, false>(P, U, d0);
        else go_tile_lo<false, false>(P, U, d0);
    }
}

void launch_tile_rminus(Pool& P, const Node* U) {
    hipLaunchKernelGGL(k_tile_rminus, dim3((unsigned)P.ntile), dim3(64 * P.tile_slices),
                       sizeof(FluxNode) * (size_t)P.tile_nodes, P.stream, mesh_view(P), (const InstDev*)P.tab, U,
                       (const double*)P.ulo_h, (const double2*)P.dmu, (const double*)P.res, P.Rm,
                       P.tune.k[KID_RMINUS].remap);
}

void launch_tile_apply(Pool& P, const Node* U, const Node* Uo, Node* out, int stage, bool bdy) {
    hipLaunchKernelGGL(k_tile_apply, dim3((unsigned)P.ntile), dim3(64 * P.tile_slices),
                       sizeof(ApplyNode) * (size_t)P.tile_nodes, P.stream, mesh_view(P), (const InstDev*)P.tab, U, Uo,
                       (const double*)P.ulo_h, (const double2*)P.ulo_q, out, (const double2*)P.dmu,
                       (const double*)P.res, (const double*)P.Rm, stage, bdy ? 1 : 0, P.flags,
                       P.tune.k[KID_APPLY].remap);
}

void launch_tile_alpha(Pool& P, const Node* U) {
    hipLaunchKernelGGL(k_tile_alpha, dim3((unsigned)P.ntile), dim3(64 * P.tile_slices),
                       sizeof(double) * (size_t)P.tile_nodes, P.stream, mesh_view(P), (const InstDev*)P.tab, U, P.alpha,
                       P.tune.k[KID_ALPHA].remap);
}

void launch_tile_dt(Pool& P, const Node* U, double* d0, double* alpha, int all, bool advance) {
    hipLaunchKernelGGL(k_tile_dt, dim3((unsigned)P.ntile), dim3(64 * P.tile_slices),
                       sizeof(DtNode) * (size_t)P.tile_nodes, P.stream, mesh_view(P), P.tab, U, d0, alpha, P.vmax,
                       P.flags, P.done, all, advance ? 1 : 0, P.ninst(), P.tune.k[KID_DT].remap);
}

static_assert(sizeof(LoNode) * kTileNodes <= 65536, "a tile's records fit a workgroup's LDS");

// The SGN records are longer than the others: pools with a longer halo keep the gather kernel.
bool tile_stage_applies(const Pool& P) {
    return tiles_apply(P) && (!P.mode.sgn || sizeof(SgnNode) * (size_t)P.tile_nodes <= 65536);
}

void launch_tile_stage(Pool& P, const Node* U, const Node* Uo, Node* out, const double* d0, bool alpha, int stage, bool bdy) {
    const Mode& md = P.mode;
    if (md.viscosity_type == SWE_GALERKIN) go_tile_first<SMB_GALERKIN>(P, U, Uo, out, d0, false, stage, bdy);
    else if (md.viscous_type == 1) go_tile_first<SMB_1>(P, U, Uo, out, d0, alpha, stage, bdy);
    else if (md.roundoff) go_tile_first<SMB_ROUNDOFF>(P, U, Uo, out, d0, alpha, stage, bdy);
    else go_tile_first<SMB_2>(P, U, Uo, out, d0, alpha, stage, bdy);
}

void launch_tile_ev(Pool& P, const Node* U, const Node* Uo, Node* out, int stage, bool bdy) {
    auto go = [&](auto src) {
        hipLaunchKernelGGL((k_tile_ev<decltype(src)::value>), dim3((unsigned)P.ntile), dim3(64 * P.tile_slices),
                           sizeof(StageNode) * (size_t)P.tile_nodes, P.stream, mesh_view(P), (const InstDev*)P.tab, U,
                           Uo, out, (const double2*)P.dmu, (const double*)P.res, P.mode.roundoff, stage, bdy ? 1 : 0,
                           P.flags, P.tune.k[KID_EV].remap);
    };
    if (P.any_src) go(std::true_type{});
    else go(std::false_type{});
}

}  // namespace swe
