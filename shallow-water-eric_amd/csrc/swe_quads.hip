// swe_quads.hip -- the tile passes of small launches: four lanes per row.  A mesh that cannot give every SIMD
// several waves is bound by the length of one wave's dependent instructions: with a lane per row a wave walks
// the up to 10 entries of its rows one after the other, each about 0.5 us of wave speed and sums.  Here lane k
// of a row's quad takes entries k, k+4, ... and evaluates their terms, and the quad then adds the terms of its
// four entries in entry order, each read from the lane that holds it (quad permutations), so every sum is the
// same sequence of additions as in swe_tiles.hip: the same bits.  A term an entry does not have is -0.0, which
// leaves any sum as it is.
//
// Tiles, staging and arguments are swe_tiles.hip's.  A workgroup has four threads per row of its tile, so one
// thread stages each row and each row of the halo.  The alpha limiter's factors are computed where a stage
// stages its nodes (from the dt pass in the first stage): a launch less, for about 1.6 times as many sums.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "swe_tile.h"

namespace swe {

namespace {

constexpr int kQuadSlices = 1;                       // largest tile these kernels take (quads_apply)
constexpr int kQuadBlock = 256 * kQuadSlices;
constexpr int kAhead = 3;                            // entries a lane loads ahead (rows of up to 12 at once)

// Value of lane K of this lane's quad.
template <int K>
__device__ __forceinline__ double quad_get(double v) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)b, K * 0x55, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(b >> 32), K * 0x55, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// s plus the terms of the quad's four entries, in entry order, each entry's in the order given.
template <int K, class... Ts>
__device__ __forceinline__ double quad_add1(double s, Ts... t) {
    ((s = s + quad_get<K>(t)), ...);
    return s;
}
template <class... Ts>
__device__ __forceinline__ double quad_add(double s, Ts... t) {
    s = quad_add1<0>(s, t...);
    s = quad_add1<1>(s, t...);
    s = quad_add1<2>(s, t...);
    return quad_add1<3>(s, t...);
}

struct QuadHead {
    int s0, nsl, inst, tid;
    int rt, k, i;         // row within the tile, lane of its quad, global row
    int len;              // entries of the row (0 past the tile)
    int64_t pb;           // first slot of the row
    int srow, slen;       // the row this thread stages (-1: none; a halo row past the list: not staged), its entries
};
__device__ __forceinline__ QuadHead quad_head(const Mesh& M, int remap) {
    QuadHead h;
    const int b = remap ? xcd_block() : (int)blockIdx.x;
    const int ts = (int)(blockDim.x >> 8), R = 64 * ts;
    h.tid = (int)threadIdx.x;
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
    h.rt = h.tid >> 2;
    h.k = h.tid & 3;
    const int w = __builtin_amdgcn_readfirstlane(h.tid >> 8);
    const bool own = w < h.nsl;
    const int sw = own ? h.s0 + w : h.s0 + h.nsl - 1;
    h.i = sw * 64 + (h.rt & 63);
    h.len = M.len[h.i];
    h.pb = M.sl[sw].sbase + (h.rt & 63);
    if (!own) h.len = 0;
    const int x = h.tid - R;
    const int hrow = M.halo[(int64_t)h.s0 * kHaloStride + ((x >= 0 && x < h.nsl * kHaloStride) ? x : 0)];
    h.srow = (x >= 0) ? (x < S.nhalo ? hrow : -1) : (h.tid < 64 * h.nsl ? h.s0 * 64 + h.tid : -1);
    h.slen = (x < 0 && h.srow >= 0) ? M.len[h.srow] : 1;
    return h;
}

// Entries k, k+4, ... of a row, kAhead of them loaded ahead: c_ij, one double2 and one double per entry as the
// pass reads them, and the column within the tile (the row itself where there is no entry).
template <bool C, bool V2, bool V1>
struct QuadRow {
    double2 c[kAhead], v2[kAhead];
    double v1[kAhead];
    int l[kAhead];
    int len, rt;
    int64_t p;            // slot of the lane's next entry
    int q;                // and its position

    __device__ __forceinline__ void fetch(int a, int64_t slot, const Mesh& M, const double2* __restrict__ x2,
                                          const double* __restrict__ x1) {
        if constexpr (C) c[a] = ld_entry(M.c + slot);
        if constexpr (V2) v2[a] = ld_entry(x2 + slot);
        if constexpr (V1) v1[a] = ld_entry1(x1 + slot);
        l[a] = M.lcol[slot];
    }
    __device__ __forceinline__ void start(const QuadHead& h, int n, const Mesh& M, const double2* __restrict__ x2,
                                          const double* __restrict__ x1) {
        len = n;
        rt = h.rt;
        q = h.k;
        p = h.pb + 64 * (int64_t)h.k;
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            c[a] = make_double2(0.0, 0.0);
            v2[a] = make_double2(0.0, 0.0);
            v1[a] = 0.0;
            l[a] = rt;
            if (q + 4 * a < len) fetch(a, p + 256 * (int64_t)a, M, x2, x1);
        }
    }
    __device__ __forceinline__ bool has() const { return q < len; }
    __device__ __forceinline__ bool more() const { return (q & ~3) < len; }      // the same on the whole quad
    __device__ __forceinline__ void next(const Mesh& M, const double2* __restrict__ x2, const double* __restrict__ x1) {
#pragma unroll
        for (int a = 0; a + 1 < kAhead; ++a) {
            c[a] = c[a + 1];
            v2[a] = v2[a + 1];
            v1[a] = v1[a + 1];
            l[a] = l[a + 1];
        }
        if (q + 4 * kAhead < len) fetch(kAhead - 1, p + 256 * (int64_t)kAhead, M, x2, x1);
        q += 4;
        p += 256;
    }
};

// =============================================================================================
// FCT / entropy-viscosity stage, pass 1: k_tile_lo's results.
// =============================================================================================
template <bool WET, bool ALPHA, bool WRITE_LO, bool D0>
__device__ __forceinline__ void quad_lo_rows(const LoNode* __restrict__ nodes, const Mesh& M,
                                             QuadRow<true, false, D0>& row, const Node& I, const Consts& K,
                                             const double* __restrict__ d0, double2* __restrict__ dmu, int roundoff,
                                             LoSums& s, int& err) {
    constexpr bool SPLIT = WRITE_LO && !WET;      // the entropy residual's ratios are not the low-order sums'
    const double nz = -0.0;
    const Rcp r16 = uniform_rcp(K.g16);
    const LoNode& A = nodes[row.rt];
    const double ovh_i = A.ovh, sql = A.sq, qi = A.q, ai = A.alpha, Ei = A.E;
    const double v1i = I.qx * ovh_i, v2i = I.qy * ovh_i;
    const double thr_lo = roundoff ? K.htiny : 0.0;
    double r1 = 0.0, r2 = 0.0, r3 = 0.0, fix = 0.0, e1 = 0.0, e2 = 0.0, e3 = 0.0, emax = 0.0, emin = 0.0;
    for (bool first = true; row.more(); first = false) {
        double f0 = nz, f1 = nz, a0 = nz, a1 = nz, a2 = nz, xe = nz, xx2 = nz, xx3 = nz, b1 = nz, b2 = nz, g1 = nz, g2 = nz;
        double y1 = nz, y2 = nz, z1 = nz, z2 = nz, w1 = nz, w2 = nz, t2 = nz, t3 = nz, Ej = Ei;
        if (row.has()) {
            const double2 c = row.c[0];
            const int l = row.l[0];
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
            const bool off = (l != row.rt);
            const double xm = -(c.x * (v1j)) - c.y * (v2j);
            xe = -(c.x * (v1j * J.h)) - c.y * (v2j * J.h);
            xx2 = -(c.x * (v1j * J.qx)) - c.y * (v2j * J.qx);
            xx3 = -(c.x * (v1j * J.qy)) - c.y * (v2j * J.qy);
            const double topo = K.g * I.h * (J.h + J.z - I.h - I.z);
            t2 = -(topo * c.x);
            t3 = -(topo * c.y);
            Ej = n.E;
            if (WRITE_LO) {
                if (roundoff) f0 = xm;
                else a0 = xe;
            }
            if (off) {
                double d = D0 ? row.v1[0] : dij_from_c(c, I, J, ovh_i, ovh_j, sql, n.sq, K, r16, err);
                double mu = mu_of(c.x, c.y, v1i, v2i, v1j, v2j);
                d = fmaxF(d, mu);
                if constexpr (ALPHA) {
                    const double a = fmaxF(ai, n.alpha);
                    d = d * a;
                    mu = mu * a;
                }
                st_entry(dmu + row.p, make_double2(d, mu));
                if (WRITE_LO) {
                    if (roundoff) {
                        f0 = -mu;
                        f1 = (d - mu) * (-ratijr);
                        a0 = (xm + mu) * J.h;
                        a1 = posF((d - mu) * Hji);
                    } else {
                        a1 = d * (J.h * ratjir - I.h * ratijr);
                        a2 = mu * (J.h * (1.0 - ratjir) - I.h * (1.0 - ratijr));
                    }
                }
                const double a = WRITE_LO ? ratjir : ratji0, b = WRITE_LO ? ratijr : ratij0;
                b1 = d * (J.qx * a - I.qx * b);
                b2 = mu * (J.qx * (1.0 - a) - I.qx * (1.0 - b));
                g1 = d * (J.qy * a - I.qy * b);
                g2 = mu * (J.qy * (1.0 - a) - I.qy * (1.0 - b));
                w1 = d * (J.h * ratji0 - I.h * ratij0);
                w2 = mu * (J.h * (1.0 - ratji0) - I.h * (1.0 - ratij0));
                if (SPLIT) {
                    y1 = d * (J.qx * ratji0 - I.qx * ratij0);
                    y2 = mu * (J.qx * (1.0 - ratji0) - I.qx * (1.0 - ratij0));
                    z1 = d * (J.qy * ratji0 - I.qy * ratij0);
                    z2 = mu * (J.qy * (1.0 - ratji0) - I.qy * (1.0 - ratij0));
                }
            }
        }
        if (WRITE_LO) {
            if (roundoff) {
                fix = quad_add(fix, f0, f1);
                r1 = quad_add(r1, a0, a1);
            } else {
                r1 = quad_add(r1, a0, a1, a2);
            }
        }
        r2 = quad_add(r2, xx2, b1, b2, t2);
        r3 = quad_add(r3, xx3, g1, g2, t3);
        e1 = quad_add(e1, xe, w1, w2);
        if (SPLIT) {
            e2 = quad_add(e2, xx2, y1, y2, t2);
            e3 = quad_add(e3, xx3, z1, z2, t3);
        }
        // (the row's own entropy in place of a missing entry's: its diagonal entry has that value too)
        const double E0 = quad_get<0>(Ej), E1 = quad_get<1>(Ej), E2 = quad_get<2>(Ej), E3 = quad_get<3>(Ej);
        if (first) emax = emin = E0;
        const auto take = [&](double E) {
            emax = (E > emax) ? E : emax;
            emin = (E < emin) ? E : emin;
        };
        take(E0);
        take(E1);
        take(E2);
        take(E3);
        row.next(M, nullptr, d0);
    }
    if (!SPLIT) {
        e2 = r2;
        e3 = r3;
    }
    s = LoSums{r1, r2, r3, fix, e1, e2, e3, emax, emin};
}

template <bool ALPHA, bool WRITE_LO, bool HAS_SRC, bool D0>
__global__ void __launch_bounds__(kQuadBlock)
k_quad_lo(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, double* __restrict__ ulo_h,
          double2* __restrict__ ulo_q, double2* __restrict__ dmu, double* __restrict__ res,
          const double* __restrict__ d0, const double* __restrict__ alpha, int roundoff, int* __restrict__ flags_out,
          int remap) {
    extern __shared__ double smem[];
    LoNode* nodes = (LoNode*)smem;
    const QuadHead h = quad_head(M, remap);
    const bool go = T[h.inst].go != 0;
    const Consts K = T[h.inst].K;
    const double dt = T[h.inst].dt;
    const int len = go ? h.len : 0;
    QuadRow<true, false, D0> row;
    row.start(h, len, M, nullptr, d0);
    const double mi = M.m[h.i];
    bool wet = true;
    if (go && h.srow >= 0) {
        const Node A = U[h.srow];
        double a = 0.0;
        if constexpr (ALPHA) a = D0 ? alpha[h.srow] : alpha_of(M, U, h.srow, A.h, K.htiny);
        nodes[h.tid] = lo_node<D0>(A, a, K);
        wet = A.h > fmaxF(K.htiny, 0.0) || h.slen == 0;
    }
    const bool all_wet = __syncthreads_and(wet ? 1 : 0) != 0;
    if (len == 0) return;
    const LoNode& A = nodes[h.rt];
    const Node I{A.h, A.qx, A.qy, A.z};
    int err = 0;
    LoSums s;
    if (all_wet) quad_lo_rows<true, ALPHA, WRITE_LO, D0>(nodes, M, row, I, K, d0, dmu, roundoff, s, err);
    else quad_lo_rows<false, ALPHA, WRITE_LO, D0>(nodes, M, row, I, K, d0, dmu, roundoff, s, err);
    if (h.k == 0) lo_finish<WRITE_LO, HAS_SRC>(I, A.ovh, A.E, s, mi, dt, K, roundoff, h.i, ulo_h, ulo_q, res, err);
    raise_flag(flags_out, h.inst, err);
}

// =============================================================================================
// FCT stage, pass 2: k_tile_rminus's R-.
// =============================================================================================
__global__ void __launch_bounds__(kQuadBlock)
k_quad_rminus(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, const double* __restrict__ ulo_h,
              const double2* __restrict__ dmu, const double* __restrict__ res, double* __restrict__ Rm, int remap) {
    extern __shared__ double smem[];
    FluxNode* nodes = (FluxNode*)smem;
    const QuadHead h = quad_head(M, remap);
    const bool go = T[h.inst].go != 0;
    const double dt = T[h.inst].dt;
    const double htiny = T[h.inst].K.htiny;
    const int len = go ? h.len : 0;
    QuadRow<false, true, false> row;
    row.start(h, len, M, dmu, nullptr);
    const double mi = M.m[h.i], hL = ulo_h[h.i];
    if (go && h.srow >= 0) {
        const Node A = U[h.srow];
        nodes[h.tid] = FluxNode{A.h, A.z, own_ratio(A.h, A.z), res[h.srow]};
    }
    __syncthreads();
    if (len == 0) return;
    const FluxNode I = nodes[h.rt];
    double P = -1.0e-15;
    while (row.more()) {
        double t = -0.0;
        if (row.has() && row.l[0] != h.rt) {
            double dA, muA, rij_, rji_;
            const double f = tile_flux(I, nodes[row.l[0]], row.v2[0], dA, muA, rij_, rji_);
            if (f < 0.0) t = f;
        }
        P = quad_add(P, t);
        row.next(M, dmu, nullptr);
    }
    const double scaled = (mi / dt) * hL;
    const double Q = 0.0 - scaled;
    double Ri = fminF(Q / P, 1.0);
    if (scaled <= htiny) Ri = 0.0;
    if (h.k == 0) Rm[h.i] = Ri;
}

// =============================================================================================
// FCT stage, pass 3: k_tile_apply's update.
// =============================================================================================
__global__ void __launch_bounds__(kQuadBlock)
k_quad_apply(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, const Node* __restrict__ Uo,
             const double* __restrict__ ulo_h, const double2* __restrict__ ulo_q, Node* __restrict__ out,
             const double2* __restrict__ dmu, const double* __restrict__ res, const double* __restrict__ Rm, int stage,
             int bdy, int* __restrict__ flags_out, int remap) {
    extern __shared__ double smem[];
    ApplyNode* nodes = (ApplyNode*)smem;
    const QuadHead h = quad_head(M, remap);
    const bool go = T[h.inst].go != 0;
    const double dt = T[h.inst].dt;
    const int check_h = T[h.inst].K.check_h;
    const int len = go ? h.len : 0;
    QuadRow<false, true, false> row;
    row.start(h, len, M, dmu, nullptr);
    const double mi = M.m[h.i], hL = ulo_h[h.i];
    const double2 qL = ulo_q[h.i];
    if (go && h.srow >= 0) {
        const Node A = U[h.srow];
        nodes[h.tid] = ApplyNode{A.h, A.z, own_ratio(A.h, A.z), res[h.srow], A.qx, A.qy, Rm[h.srow], 0.0};
    }
    __syncthreads();
    if (len == 0) return;
    const ApplyNode I = nodes[h.rt];
    double x1 = 0.0, x2 = 0.0, x3 = 0.0;
    while (row.more()) {
        double a1 = -0.0, a2 = -0.0, b1 = -0.0, b2 = -0.0, c1 = -0.0, c2 = -0.0;
        if (row.has() && row.l[0] != h.rt) {
            const ApplyNode& J = nodes[row.l[0]];
            double dA, muA, ratij, ratji;
            const double f = tile_flux(I, J, row.v2[0], dA, muA, ratij, ratji);
            const double lim = (f >= 0.0) ? J.Rm : I.Rm;
            const double d = dA * lim;
            const double mu = muA * lim;
            const double a = 1.0 - ratji, b = 1.0 - ratij;
            a1 = d * (J.h * ratji - I.h * ratij);
            a2 = mu * (J.h * a - I.h * b);
            b1 = d * (J.qx * ratji - I.qx * ratij);
            b2 = mu * (J.qx * a - I.qx * b);
            c1 = d * (J.qy * ratji - I.qy * ratij);
            c2 = mu * (J.qy * a - I.qy * b);
        }
        x1 = quad_add(x1, a1, a2);
        x2 = quad_add(x2, b1, b2);
        x3 = quad_add(x3, c1, c2);
        row.next(M, dmu, nullptr);
    }
    if (h.k != 0) return;
    Node o{hL + dt * (x1 / mi), qL.x + dt * (x2 / mi), qL.y + dt * (x3 / mi), I.z};
    const int err = (check_h && o.h < 0.0) ? FLAG_NEG_H : 0;
    stage_out(o, M, T[h.inst], Uo, out, h.i, stage, bdy);
    raise_flag(flags_out, h.inst, err);
}

// =============================================================================================
// First-order stage and the entropy-viscosity update: k_tile_stage's and k_tile_ev's.
// =============================================================================================
// Terms of an entry for the low-order sums (stage_entry's additions, in order).
struct QuadTerms {
    double f0 = -0.0, f1 = -0.0, t[3][4] = {{-0.0, -0.0, -0.0, -0.0}, {-0.0, -0.0, -0.0, -0.0}, {-0.0, -0.0, -0.0, -0.0}};
};
template <int SMB>
__device__ __forceinline__ void quad_terms(QuadTerms& w, const Node& I, const Node& J, const double2 c, double v1i,
                                           double v2i, double v1j, double v2j, double Hij, double Hji, double ratij,
                                           double ratji, double d, double mu, bool off, const Consts& K) {
    const double ui[3] = {I.h, I.qx, I.qy}, uj[3] = {J.h, J.qx, J.qy};
    if constexpr (SMB == SMB_1) {
        const double t = 0.5 * K.g * (Hji * Hji - Hij * Hij);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            w.t[k][0] = -(c.x * (v1j * uj[k] * ratji + v1i * ui[k] * ratij)) -
                        c.y * (v2j * uj[k] * ratji + v2i * ui[k] * ratij);
            if (off) w.t[k][1] = d * (uj[k] * ratji - ui[k] * ratij);
        }
        if (off) {
            w.t[1][3] = -(t * c.x);
            w.t[2][3] = -(t * c.y);
        }
    } else {
        constexpr int k0 = (SMB == SMB_ROUNDOFF) ? 1 : 0;
        if constexpr (SMB == SMB_ROUNDOFF) {
            const double xm = -(c.x * (v1j)) - c.y * (v2j);
            w.f0 = off ? -mu : xm;
            if (off) {
                w.f1 = (d - mu) * (-ratij);
                w.t[0][0] = (xm + mu) * uj[0];
                w.t[0][1] = posF((d - mu) * Hji);
            }
        }
        const double aj = 1.0 - ratji, ai = 1.0 - ratij;
#pragma unroll
        for (int k = k0; k < 3; ++k) {
            w.t[k][0] = -(c.x * (v1j * uj[k])) - c.y * (v2j * uj[k]);
            if (SMB != SMB_GALERKIN && off) {
                w.t[k][1] = d * (uj[k] * ratji - ui[k] * ratij);
                w.t[k][2] = mu * (uj[k] * aj - ui[k] * ai);
            }
        }
        const double topo = K.g * ui[0] * (uj[0] + J.z - ui[0] - I.z);
        w.t[1][3] = -(topo * c.x);
        w.t[2][3] = -(topo * c.y);
    }
}
template <int SMB>
__device__ __forceinline__ void quad_sums(double (&r)[3], double& fix, const QuadTerms& w) {
    if constexpr (SMB == SMB_ROUNDOFF) {
        fix = quad_add(fix, w.f0, w.f1);
        r[0] = quad_add(r[0], w.t[0][0], w.t[0][1]);
    } else {
        r[0] = quad_add(r[0], w.t[0][0], w.t[0][1], w.t[0][2]);
    }
    r[1] = quad_add(r[1], w.t[1][0], w.t[1][1], w.t[1][2], w.t[1][3]);
    r[2] = quad_add(r[2], w.t[2][0], w.t[2][1], w.t[2][2], w.t[2][3]);
}

template <int SMB, bool ALPHA, bool HAS_SRC, bool D0>
__global__ void __launch_bounds__(kQuadBlock)
k_quad_stage(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, const Node* __restrict__ Uo,
             Node* __restrict__ out, const double* __restrict__ d0, const double* __restrict__ alpha, int stage, int bdy,
             int* __restrict__ flags_out, int remap) {
    constexpr bool VISC = SMB != SMB_GALERKIN;
    extern __shared__ double smem[];
    StageNode* nodes = (StageNode*)smem;
    const QuadHead h = quad_head(M, remap);
    const bool go = T[h.inst].go != 0;
    const Consts K = T[h.inst].K;
    const double dt = T[h.inst].dt;
    const int len = go ? h.len : 0;
    QuadRow<true, false, VISC && D0> row;
    row.start(h, len, M, nullptr, d0);
    const double mi = M.m[h.i];
    if (go && h.srow >= 0) {
        const Node A = U[h.srow];
        double a = 0.0;
        if constexpr (ALPHA) a = D0 ? alpha[h.srow] : alpha_of(M, U, h.srow, A.h, K.htiny);
        nodes[h.tid] = StageNode{A.h, A.z, A.qx, A.qy, ovh_of(A.h, K.htiny),
                                 (VISC && !D0) ? sqrt_rn(K.g * fabs(A.h)) : 0.0, own_ratio(A.h, A.z), a};
    }
    __syncthreads();
    if (len == 0) return;
    const Rcp r16 = uniform_rcp(K.g16);
    const StageNode A = nodes[h.rt];
    const Node I{A.h, A.qx, A.qy, A.z};
    const double v1i = I.qx * A.ovh, v2i = I.qy * A.ovh;
    const double thr = (SMB == SMB_ROUNDOFF || SMB == SMB_1) ? K.htiny : 0.0;
    double r[3] = {0.0, 0.0, 0.0}, fix = 0.0;
    int err = 0;
    while (row.more()) {
        QuadTerms w;
        if (row.has()) {
            const double2 c = row.c[0];
            const int l = row.l[0];
            const StageNode& B = nodes[l];
            const Node J{B.h, B.qx, B.qy, B.z};
            const double v1j = J.qx * B.ovh, v2j = J.qy * B.ovh;
            double Hij, Hji, ratij, ratji;
            depth_ratios(I.h, I.z, A.q, J.h, J.z, B.q, Hij, Hji, ratij, ratji);
            ratij = (I.h <= thr) ? 0.0 : ratij;
            ratji = (J.h <= thr) ? 0.0 : ratji;
            const bool off = (l != h.rt);
            double d = 0.0, mu = 0.0;
            if (VISC && off) {
                d = D0 ? row.v1[0] : dij_from_c(c, I, J, A.ovh, B.ovh, A.sq, B.sq, K, r16, err);
                mu = mu_of(c.x, c.y, v1i, v2i, v1j, v2j);
                d = fmaxF(d, mu);
                if constexpr (ALPHA) {
                    const double a = fmaxF(A.alpha, B.alpha);
                    d = d * a;
                    mu = mu * a;
                }
            }
            quad_terms<SMB>(w, I, J, c, v1i, v2i, v1j, v2j, Hij, Hji, ratij, ratji, d, mu, off, K);
        }
        quad_sums<SMB>(r, fix, w);
        row.next(M, nullptr, d0);
    }
    raise_flag(flags_out, h.inst, err);
    if (h.k != 0) return;
    add_sources<HAS_SRC>(K.src, I, mi, v1i, v2i, dt, K, r[1], r[2]);
    for (int k = 0; k < 3; ++k) r[k] = r[k] / mi;
    const Node o{stage_depth<SMB>(I.h, dt, fix, mi, r[0]), I.qx + dt * r[1], I.qy + dt * r[2], I.z};
    stage_out(o, M, T[h.inst], Uo, out, h.i, stage, bdy);
}

template <int SMB, bool HAS_SRC>
__global__ void __launch_bounds__(kQuadBlock)
k_quad_ev(Mesh M, const InstDev* __restrict__ T, const Node* __restrict__ U, const Node* __restrict__ Uo,
          Node* __restrict__ out, const double2* __restrict__ dmu, const double* __restrict__ res, int stage, int bdy,
          int* __restrict__ flags_out, int remap) {
    extern __shared__ double smem[];
    StageNode* nodes = (StageNode*)smem;     // alpha holds the residual, sq is unused
    const QuadHead h = quad_head(M, remap);
    const bool go = T[h.inst].go != 0;
    const Consts K = T[h.inst].K;
    const double dt = T[h.inst].dt;
    const int len = go ? h.len : 0;
    QuadRow<true, true, false> row;
    row.start(h, len, M, dmu, nullptr);
    const double mi = M.m[h.i];
    if (go && h.srow >= 0) {
        const Node A = U[h.srow];
        nodes[h.tid] = StageNode{A.h, A.z, A.qx, A.qy, ovh_of(A.h, K.htiny), 0.0, own_ratio(A.h, A.z), res[h.srow]};
    }
    __syncthreads();
    if (len == 0) return;
    const StageNode A = nodes[h.rt];
    const Node I{A.h, A.qx, A.qy, A.z};
    const double v1i = I.qx * A.ovh, v2i = I.qy * A.ovh;
    const double thr = (SMB == SMB_ROUNDOFF) ? K.htiny : 0.0;
    double r[3] = {0.0, 0.0, 0.0}, fix = 0.0;
    while (row.more()) {
        QuadTerms w;
        if (row.has()) {
            const double2 c = row.c[0], lo = row.v2[0];
            const int l = row.l[0];
            const StageNode& B = nodes[l];
            const Node J{B.h, B.qx, B.qy, B.z};
            const double v1j = J.qx * B.ovh, v2j = J.qy * B.ovh;
            double Hij, Hji, ratij, ratji;
            depth_ratios(I.h, I.z, A.q, J.h, J.z, B.q, Hij, Hji, ratij, ratji);
            ratij = (I.h <= thr) ? 0.0 : ratij;
            ratji = (J.h <= thr) ? 0.0 : ratji;
            const bool off = (l != h.rt);
            double d = 0.0, mu = 0.0;
            if (off) {
                const double rij = fmaxF(A.alpha, B.alpha);
                d = fminF(lo.x, 1.0 * rij);
                mu = fminF(lo.y, 1.0 * rij);
            }
            quad_terms<SMB>(w, I, J, c, v1i, v2i, v1j, v2j, Hij, Hji, ratij, ratji, d, mu, off, K);
        }
        quad_sums<SMB>(r, fix, w);
        row.next(M, dmu, nullptr);
    }
    if (h.k != 0) return;
    add_sources<HAS_SRC>(K.src, I, mi, v1i, v2i, dt, K, r[1], r[2]);
    for (int k = 0; k < 3; ++k) r[k] = r[k] / mi;
    const Node o{stage_depth<SMB>(I.h, dt, fix, mi, r[0]), I.qx + dt * r[1], I.qy + dt * r[2], I.z};
    const int err = (K.check_h && o.h < 0.0) ? FLAG_NEG_H : 0;
    stage_out(o, M, T[h.inst], Uo, out, h.i, stage, bdy);
    raise_flag(flags_out, h.inst, err);
}

// =============================================================================================
// COMPUTE_DT: k_tile_dt's d_ij, maxima and bookkeeping.
// =============================================================================================
__global__ void __launch_bounds__(kQuadBlock)
k_quad_dt(Mesh M, InstDev* __restrict__ T, const Node* __restrict__ U, double* __restrict__ d0,
          double* __restrict__ alpha, unsigned long long* __restrict__ vmax, int* __restrict__ flags,
          unsigned* __restrict__ done, int all, int advance, int ninst, int remap) {
    extern __shared__ double smem[];
    DtNode* nodes = (DtNode*)smem;
    __shared__ unsigned long long red[kQuadBlock / 64];
    __shared__ int last;
    const QuadHead h = quad_head(M, remap);
    // (per wave: a check raised meanwhile may end some waves' part; every barrier is met by all of them)
    const bool live = all ? T[h.inst].state != INST_FREE : takes_steps(T[h.inst], flags[h.inst]);
    const int len = live ? h.len : 0;
    const Consts K = T[h.inst].K;
    QuadRow<true, false, false> row;
    row.start(h, len, M, nullptr, nullptr);
    const double mi = M.m[h.i];
    if (h.srow >= 0) {
        const Node A = U[h.srow];
        nodes[h.tid] = DtNode{A.h, A.qx, A.qy, ovh_of(A.h, K.htiny), sqrt_rn(K.g * fabs(A.h)), 0.0};
    }
    __syncthreads();
    double v = 0.0;
    int err = 0;
    if (len > 0) {
        const Rcp r16 = uniform_rcp(K.g16);
        const DtNode A = nodes[h.rt];
        const Node I{A.h, A.qx, A.qy, 0.0};
        double s = 0.0, num = 0.0, den = 0.0;
        while (row.more()) {
            double d = -0.0, hj = -0.0, hi = -0.0, dh = -0.0;
            if (row.has()) {
                const int l = row.l[0];
                const DtNode& B = nodes[l];
                const Node J{B.h, B.qx, B.qy, 0.0};
                hj = J.h;
                hi = -I.h;
                dh = fabs(J.h - I.h);
                if (l != h.rt) {
                    d = dij_from_c(row.c[0], I, J, A.ovh, B.ovh, A.sq, B.sq, K, r16, err);
                    if (d0) st_entry1(d0 + row.p, d);
                }
            }
            s = quad_add(s, d);
            if (alpha) {
                num = quad_add(num, hj, hi);
                den = quad_add(den, dh);
            }
            row.next(M, nullptr, nullptr);
        }
        v = fabs(-s) / mi;
        if (alpha && h.k == 0) alpha[h.i] = alpha_value(num, den, I.h, K.htiny);
    }
    dt_finish(T, v, err, h.inst, vmax, flags, done, red, &last, advance, ninst);
}

dim3 quad_grid(const Pool& P) { return dim3((unsigned)P.ntile); }
dim3 quad_block(const Pool& P) { return dim3(256u * (unsigned)P.tile_slices); }

template <class N>
size_t quad_lds(const Pool& P) { return sizeof(N) * (size_t)P.tile_nodes; }

// f(std::bool_constant...) for run-time switches
template <class F>
void on_bools(F&& f) { f(); }
template <class F, class... B>
void on_bools(F&& f, bool b, B... rest) {
    if (b) on_bools([&](auto... x) { f(std::true_type{}, x...); }, rest...);
    else on_bools([&](auto... x) { f(std::false_type{}, x...); }, rest...);
}

template <int SMB>
void go_quad_stage(Pool& P, const Node* U, const Node* Uo, Node* out, const double* d0, bool alpha, int stage, bool bdy) {
    constexpr bool visc = SMB != SMB_GALERKIN;
    on_bools(
        [&](auto a, auto src, auto has_d0) {
            constexpr bool A = visc && decltype(a)::value, S = decltype(src)::value, D = visc && decltype(has_d0)::value;
            hipLaunchKernelGGL((k_quad_stage<SMB, A, S, D>), quad_grid(P), quad_block(P), quad_lds<StageNode>(P), P.stream,
                               mesh_view(P), (const InstDev*)P.tab, U, Uo, out, d0, (const double*)P.alpha, stage,
                               bdy ? 1 : 0, P.flags, P.tune.k[KID_STAGE_LO].remap);
        },
        alpha, P.any_src, d0 != nullptr);
}

}  // namespace

static_assert(kQuadSlices <= kMaxTileSlices && kHaloStride <= 3 * 64, "a quad workgroup has a thread per staged row");

// Pools whose tiles are one slice (tile_slices_for: up to 49,152 rows, three workgroups per CU).  Measured per
// step, a lane per row in the tiles used otherwise against four in one-slice tiles: FCT with alpha 93.6 -> 64.5 us at
// 5k nodes, 102.7 -> 80.8 at 32k, 108.3 -> 103.3 at 47k; first order 49.1 -> 34.1, 52.7 -> 42.1, 54.3 -> 47.8;
// entropy viscosity 70.6 -> 51.6, 77.2 -> 65.5, 82.9 -> 83.2.  Above, where the SIMDs have waves anyway, the
// registers of the terms and the additions made four times cost more than they give: at 50k FCT 110.2 -> 112.9 us,
// first order 55.2 -> 55.5, entropy viscosity 84.2 -> 96.5; at 100k, in two-slice tiles, FCT 133.6 -> 202.8.
bool quads_apply(const Pool& P) { return P.tile_slices <= kQuadSlices; }

void launch_quad_lo(Pool& P, const Node* U, const double* d0, bool alpha, bool write_lo) {
    on_bools(
        [&](auto a, auto w, auto src, auto has_d0) {
            constexpr bool A = decltype(a)::value, W = decltype(w)::value, S = decltype(src)::value,
                           D = decltype(has_d0)::value;
            hipLaunchKernelGGL((k_quad_lo<A, W, S, D>), quad_grid(P), quad_block(P), quad_lds<LoNode>(P), P.stream,
                               mesh_view(P), (const InstDev*)P.tab, U, P.ulo_h, P.ulo_q, P.dmu, P.res, d0,
                               (const double*)P.alpha, P.mode.roundoff, P.flags, P.tune.k[KID_FCT_LO].remap);
        },
        alpha, write_lo, P.any_src, d0 != nullptr);
}

void launch_quad_rminus(Pool& P, const Node* U) {
    hipLaunchKernelGGL(k_quad_rminus, quad_grid(P), quad_block(P), quad_lds<FluxNode>(P), P.stream, mesh_view(P),
                       (const InstDev*)P.tab, U, (const double*)P.ulo_h, (const double2*)P.dmu, (const double*)P.res, P.Rm,
                       P.tune.k[KID_RMINUS].remap);
}

void launch_quad_apply(Pool& P, const Node* U, const Node* Uo, Node* out, int stage, bool bdy) {
    hipLaunchKernelGGL(k_quad_apply, quad_grid(P), quad_block(P), quad_lds<ApplyNode>(P), P.stream, mesh_view(P),
                       (const InstDev*)P.tab, U, Uo, (const double*)P.ulo_h, (const double2*)P.ulo_q, out,
                       (const double2*)P.dmu, (const double*)P.res, (const double*)P.Rm, stage, bdy ? 1 : 0, P.flags,
                       P.tune.k[KID_APPLY].remap);
}

void launch_quad_stage(Pool& P, const Node* U, const Node* Uo, Node* out, const double* d0, bool alpha, int stage, bool bdy) {
    const Mode& md = P.mode;
    if (md.viscosity_type == SWE_GALERKIN) go_quad_stage<SMB_GALERKIN>(P, U, Uo, out, nullptr, false, stage, bdy);
    else if (md.viscous_type == 1) go_quad_stage<SMB_1>(P, U, Uo, out, d0, alpha, stage, bdy);
    else if (md.roundoff) go_quad_stage<SMB_ROUNDOFF>(P, U, Uo, out, d0, alpha, stage, bdy);
    else go_quad_stage<SMB_2>(P, U, Uo, out, d0, alpha, stage, bdy);
}

void launch_quad_ev(Pool& P, const Node* U, const Node* Uo, Node* out, int stage, bool bdy) {
    on_bools(
        [&](auto round, auto src) {
            constexpr int SMB = decltype(round)::value ? SMB_ROUNDOFF : SMB_2;
            hipLaunchKernelGGL((k_quad_ev<SMB, decltype(src)::value>), quad_grid(P), quad_block(P), quad_lds<StageNode>(P),
                               P.stream, mesh_view(P), (const InstDev*)P.tab, U, Uo, out, (const double2*)P.dmu,
                               (const double*)P.res, stage, bdy ? 1 : 0, P.flags, P.tune.k[KID_EV].remap);
        },
        P.mode.roundoff != 0, P.any_src);
}

void launch_quad_dt(Pool& P, const Node* U, double* d0, double* alpha, int all, bool advance) {
    hipLaunchKernelGGL(k_quad_dt, quad_grid(P), quad_block(P), quad_lds<DtNode>(P), P.stream, mesh_view(P), P.tab, U, d0,
                       alpha, P.vmax, P.flags, P.done, all, advance ? 1 : 0, P.ninst(), P.tune.k[KID_DT].remap);
}

}  // namespace swe
