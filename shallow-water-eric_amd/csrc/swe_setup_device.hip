// swe_setup_device.hip -- the P1 set-up of construct_matrices (SOURCES/update.f90:18-132) on the
// GPU: the pattern of st_csr (SFEMaNS/FEMSUB/st_sparsekit.f90:788-863), the consistent mass of
// qs_00_M (SFEMaNS/FEMSUB_OBJET/fem_sparsekit.f90:31-51), c_ij (update.f90:106-124), the lumped
// mass (update.f90:35-38) and the diagonal positions.
//
// Same contract as the host assembly in swe_setup.cpp, bit for bit: every entry is accumulated in
// ascending element order (Gauss points in order inside an element) with the shared element
// geometry of swe_p1.h, and lumped(i) is the sequential row sum:
//   1. node -> element lists: counts (integer atomics), exclusive scan, fill, then each list
//      sorted ascending in its lane, so the lists do not depend on the order the atomics ran in;
//   2. row pattern: the sorted unique nodes of the row's elements, counted, scanned into ia, written to ja;
//   3. values: mass and c_ij accumulated element by element, eight lanes per row, then lumped.
// A node may belong to at most kMaxElems elements (rows of at most 3*kMaxElems candidates);
// larger fans are reported as SWE_EINVAL and can be assembled on the host.
#include <hip/hip_runtime.h>
#include <hipcub/device/device_radix_sort.hpp>
#include <hipcub/device/device_scan.hpp>

#include <cmath>
#include <cstdint>
#include <cstring>

#include "swe_amd.h"
#include "swe_engine.h"
#include "swe_p1.h"

namespace {

constexpr int kMaxElems = 32;
constexpr int kMaxPattern = 3 * kMaxElems;

using swe_p1::ElemGeom;
using swe_p1::P1Rule;
using swe_p1::element_geometry;

constexpr int kFlagMany = 1, kFlagRange = 2;   // a node in more than kMaxElems elements; an entry of jj out of range

__global__ void k_count_elems(const int* __restrict__ jj, int64_t n3, int np, int64_t* __restrict__ cnt,
                              unsigned long long* __restrict__ flag) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n3) return;
    const int j = jj[q];
    if (j < 1 || j > np) atomicOr(flag, (unsigned long long)kFlagRange);
    else atomicAdd((unsigned long long*)&cnt[j - 1], 1ull);
}

__global__ void k_fill_elems(const int* __restrict__ jj, int me, int np, const int64_t* __restrict__ start,
                             int* __restrict__ fill, int* __restrict__ elem) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= 3 * (int64_t)me) return;
    const int n = jj[q] - 1;
    if (n < 0 || n >= np) return;
    const int k = atomicAdd(&fill[n], 1);
    elem[start[n] + k] = (int)(q / 3);
}

// A lane's array of N ints in LDS (word t of lane l at t*64 + l: no bank conflicts).  As a private array it would
// lie in scratch memory, each access a trip through the caches.
struct LaneInts {
    int* base;
    __device__ int& operator[](int t) const { return base[64 * t]; }
};

// Sorted unique nodes (0-based) of the n elements el; returns their number.
__device__ int row_pattern(LaneInts el, int n, const int* __restrict__ jj, LaneInts row) {
    int w = 0;
    for (int s = 0; s < n; ++s) {
        const int m = el[s];
        for (int a = 0; a < 3; ++a) {
            const int v = jj[3 * (int64_t)m + a] - 1;
            // insert v keeping row[0..w) sorted and unique
            int c = w - 1, x = -1;
            while (c >= 0 && (x = row[c]) > v) --c;
            if (c >= 0 && x == v) continue;
            for (int t = w; t > c + 1; --t) row[t] = row[t - 1];
            row[c + 1] = v;
            ++w;
        }
    }
    return w;
}

// One wave per 64 rows.  FILL false: sorts each row's element list ascending (elem) and counts its pattern (cnt);
// flags a node in more than kMaxElems elements.  FILL true: writes the pattern (ja) and the diagonal's position.
template <bool FILL>
__global__ void __launch_bounds__(64)
k_row_pattern(int np, const int64_t* __restrict__ start, int* __restrict__ elem, const int* __restrict__ jj,
              int64_t* __restrict__ cnt, unsigned long long* __restrict__ flag, const int64_t* __restrict__ ia0,
              int* __restrict__ ja, int* __restrict__ diag) {
    __shared__ int lds[64 * (kMaxElems + kMaxPattern)];
    const LaneInts el{lds + threadIdx.x}, row{lds + 64 * kMaxElems + threadIdx.x};
    const int i = (int)(blockIdx.x * 64 + threadIdx.x);
    if (i >= np) return;
    const int64_t b = start[i];
    const int n = (int)(start[i + 1] - b);
    if (n > kMaxElems) {
        if (!FILL) {
            atomicOr(flag, (unsigned long long)kFlagMany);
            cnt[i] = 0;
        }
        return;
    }
    for (int a = 0; a < n; ++a) {
        const int v = elem[b + a];
        int c = a - 1, x;
        while (!FILL && c >= 0 && (x = el[c]) > v) {
            el[c + 1] = x;
            --c;
        }
        el[FILL ? a : c + 1] = v;
    }
    const int w = row_pattern(el, n, jj, row);
    if (!FILL) {
        for (int a = 0; a < n; ++a) elem[b + a] = el[a];
        cnt[i] = w;
    } else {
        const int64_t p0 = ia0[i];
        for (int q = 0; q < w; ++q) {
            const int j = row[q];
            ja[p0 + q] = j + 1;
            if (j == i) diag[i] = (int)(p0 + q) + 1;
        }
    }
}

// mass, c_ij and lumped of the rows: eight lanes per row, lane e taking the entries e, e+8, ...; an entry walks
// the row's elements in ascending order and adds what those that contain its column give, as the host does
// (qs_00_M visits l, then nj, then ni; x(d) = SUM_l dw(d,nj,l) * ww(ni,l) * rj(l)), so the sums are the same
// additions.  (One lane per row, finding the pattern and adding into
// the entries in memory: 631 us at 300k nodes; the pattern and these values now 119 + 144.)
__global__ void __launch_bounds__(256)
k_row_values(int np, const int64_t* __restrict__ start, const int* __restrict__ elem, const int* __restrict__ jj,
             const double* __restrict__ rr, const int64_t* __restrict__ ia0, const int* __restrict__ ja,
             double* __restrict__ mass, double* __restrict__ lumped, double* __restrict__ cx, double* __restrict__ cy) {
    const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 3), e = (int)(threadIdx.x & 7);
    if (i >= np) return;
    const P1Rule R;
    const int64_t p0 = ia0[i], s0 = start[i], s1 = start[i + 1];
    const int n = (int)(ia0[i + 1] - p0);
    double sl = 0.0;
    for (int q0 = 0; q0 < n; q0 += 8) {
        const bool has = q0 + e < n;
        double am = 0.0, ax = 0.0, ay = 0.0;
        if (has) {
            const int64_t p = p0 + q0 + e;
            const int j = ja[p] - 1;
            for (int64_t s = s0; s < s1; ++s) {
                const int64_t m = elem[s];
                const int nd[3] = {jj[3 * m] - 1, jj[3 * m + 1] - 1, jj[3 * m + 2] - 1};
                if (nd[0] != j && nd[1] != j && nd[2] != j) continue;
                const int ni = (nd[0] == i) ? 0 : (nd[1] == i) ? 1 : 2;
                ElemGeom G;
                element_geometry(R, rr, nd, G);
                double wi[3];
#pragma unroll
                for (int l = 0; l < 3; ++l) wi[l] = (ni == 0) ? R.ww[0][l] : (ni == 1) ? R.ww[1][l] : R.ww[2][l];
#pragma unroll
                for (int l = 0; l < 3; ++l) {
                    const double al = 1.0 * G.rj[l];
#pragma unroll
                    for (int nj = 0; nj < 3; ++nj)
                        if (nd[nj] == j) am = am + R.ww[nj][l] * al * wi[l];
                }
#pragma unroll
                for (int nj = 0; nj < 3; ++nj)
                    if (nd[nj] == j) {
                        double x[2];
#pragma unroll
                        for (int d = 0; d < 2; ++d) {
                            double sacc = 0.0;
#pragma unroll
                            for (int l = 0; l < 3; ++l) sacc = sacc + G.dw[d][nj][l] * wi[l] * G.rj[l];
                            x[d] = sacc;
                        }
                        ax = ax + x[0];
                        ay = ay + x[1];
                    }
            }
            mass[p] = am;
            cx[p] = ax;
            cy[p] = ay;
        }
        const int left = (n - q0 < 8) ? n - q0 : 8;
        for (int k = 0; k < left; ++k) sl = sl + __shfl(am, k, 8);
    }
    if (e == 0) lumped[i] = sl;
}

unsigned grid_of(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

struct swe_assembly {
    int np = 0;
    int64_t nnz = 0;
    hipStream_t stream = nullptr;
    void *nodes = nullptr, *entries = nullptr;   // the allocations that hold the arrays per node and per entry
    int64_t* ia0 = nullptr;   // 0-based row starts, np+1
    int* ja = nullptr;
    int* diag = nullptr;
    double *mass = nullptr, *lumped = nullptr, *cx = nullptr, *cy = nullptr;
    double* rr = nullptr;     // node coordinates rr(2,np), kept for the locality order of the layout
};

namespace {

// Device memory of the set-up is stream-ordered (hipMallocAsync / hipFreeAsync on the set-up's own
// stream): unlike hipFree, releasing it does not wait for the work queued on other streams, so a
// batch can admit meshes while its steps run.  Each stage takes one block for all its arrays.
hipError_t block_alloc(swe::Carver& c, void** block, hipStream_t s) {
    const hipError_t e = hipMallocAsync(block, c.bytes() ? c.bytes() : 1, s);
    if (e == hipSuccess) c.place(*block);
    else *block = nullptr;
    return e;
}

void dfree(void* p, hipStream_t s) {
    if (p) (void)hipFreeAsync(p, s);
}

void release(swe_assembly* a) {
    if (!a) return;
    dfree(a->nodes, a->stream);
    dfree(a->entries, a->stream);
    if (a->stream) {
        (void)hipStreamSynchronize(a->stream);
        (void)hipStreamDestroy(a->stream);
    }
    delete a;
}

// Scratch of an exclusive prefix sum of n values, and the sum itself on stream s (nothing waits here).
size_t scan_bytes(int n) {
    size_t bytes = 0;
    (void)hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, (const int64_t*)nullptr, (int64_t*)nullptr, n, nullptr);
    return bytes;
}
hipError_t exclusive_scan(const int64_t* in, int64_t* out, int n, char* tmp, size_t bytes, hipStream_t s) {
    return hipcub::DeviceScan::ExclusiveSum(tmp, bytes, in, out, n, s);
}

}  // namespace

extern "C" int swe_assemble_device(int np, int me, const int* jj, const double* rr, swe_assembly** out,
                                   long long* nnz) {
    swe::clear_error();
    if (!out || !nnz || !jj || !rr || np <= 0 || me <= 0) return swe::fail(SWE_EINVAL, "null or empty argument");
    *out = nullptr;
    *nnz = 0;
    const int64_t n3 = 3 * (int64_t)me;
    swe_assembly* a = new swe_assembly();
    a->np = np;
    int *djj = nullptr, *elem = nullptr, *fill = nullptr;
    unsigned long long* flag = nullptr;
    int64_t *cnt = nullptr, *start = nullptr;
    char* tmp = nullptr;
    void* work = nullptr;
    hipError_t e = hipStreamCreateWithFlags(&a->stream, hipStreamNonBlocking);
    hipStream_t s = a->stream;
    const size_t nscan = scan_bytes(np + 1);
    swe::Carver keep, temp;
    keep.add(&a->rr, 2 * (size_t)np);
    keep.add(&a->ia0, (size_t)np + 1);
    keep.add(&a->diag, (size_t)np);
    keep.add(&a->lumped, (size_t)np);
    temp.add(&flag, 1);          // flag, cnt and fill start at zero: one clearing
    temp.add(&cnt, (size_t)np + 1);
    temp.add(&fill, (size_t)np);
    const size_t zeroed = temp.bytes();
    temp.add(&djj, (size_t)n3);
    temp.add(&elem, (size_t)n3);
    temp.add(&start, (size_t)np + 1);
    temp.add(&tmp, nscan);
    if (e == hipSuccess) e = block_alloc(keep, &a->nodes, s);
    if (e == hipSuccess) e = block_alloc(temp, &work, s);
    if (e == hipSuccess) e = hipMemcpyAsync(djj, jj, sizeof(int) * (size_t)n3, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemcpyAsync(a->rr, rr, sizeof(double) * 2 * (size_t)np, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemsetAsync(work, 0, zeroed, s);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_count_elems, dim3(grid_of(n3, 256)), dim3(256), 0, s, djj, n3, np, cnt, flag);
        e = exclusive_scan(cnt, start, np + 1, tmp, nscan, s);
    }
    unsigned long long bad = 0;
    int64_t total = 0;
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_fill_elems, dim3(grid_of(n3, 256)), dim3(256), 0, s, djj, me, np, start, fill, elem);
        // (cnt's last word stays the zero it was: no entry of jj counts there)
        hipLaunchKernelGGL(k_row_pattern<false>, dim3(grid_of(np, 64)), dim3(64), 0, s, np, start, elem, djj, cnt, flag,
                           (const int64_t*)nullptr, (int*)nullptr, (int*)nullptr);
        e = exclusive_scan(cnt, a->ia0, np + 1, tmp, nscan, s);
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&bad, flag, sizeof bad, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipMemcpyAsync(&total, a->ia0 + np, sizeof total, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    int rc = SWE_OK;
    if (e != hipSuccess || (bad & kFlagRange)) {
        // (also where the device failed: an entry out of range is refused as such on any machine)
        for (int64_t q = 0; q < n3 && rc == SWE_OK; ++q)
            if (jj[q] < 1 || jj[q] > np) rc = swe::fail(SWE_EINVAL, "jj(%lld)=%d out of range", (long long)q + 1, jj[q]);
    } else if (e == hipSuccess && bad) {
        rc = swe::fail(SWE_EINVAL, "a node belongs to more than %d elements; use swe_assemble", kMaxElems);
    } else if (e == hipSuccess && total >= (int64_t)INT32_MAX) {
        rc = swe::fail(SWE_EINVAL, "nnz = %lld does not fit the 32-bit row pointers", (long long)total);
    } else if (e == hipSuccess) {
        a->nnz = total;
        swe::Carver entries;
        entries.add(&a->ja, (size_t)total);
        entries.add(&a->mass, (size_t)total);
        entries.add(&a->cx, (size_t)total);
        entries.add(&a->cy, (size_t)total);
        e = block_alloc(entries, &a->entries, s);
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_row_pattern<true>, dim3(grid_of(np, 64)), dim3(64), 0, s, np, start, elem, djj,
                               (int64_t*)nullptr, flag, (const int64_t*)a->ia0, a->ja, a->diag);
            hipLaunchKernelGGL(k_row_values, dim3(grid_of(8 * (int64_t)np, 256)), dim3(256), 0, s, np, start, elem, djj,
                               (const double*)a->rr, (const int64_t*)a->ia0, (const int*)a->ja, a->mass, a->lumped, a->cx,
                               a->cy);
            e = hipGetLastError();
        }
        if (e == hipSuccess) e = hipStreamSynchronize(s);
    }
    dfree(work, s);
    if (e != hipSuccess && rc == SWE_OK) rc = swe::fail(SWE_EHIP, "device assembly: %s", hipGetErrorString(e));
    if (rc != SWE_OK) {
        release(a);
        return rc;
    }
    *out = a;
    *nnz = (long long)a->nnz;
    return SWE_OK;
}

extern "C" int swe_assembly_get(swe_assembly* a, int* ia, int* ja, int* diag, double* mass, double* lumped,
                                double* cx, double* cy) {
    if (!a) return swe::fail(SWE_EINVAL, "null assembly");
    const size_t nz = (size_t)a->nnz, np = (size_t)a->np;
    hipStream_t s = a->stream;
    hipError_t e = hipSuccess;
    if (ia) {
        // 1-based 32-bit row pointers, as st_csr builds them
        int64_t* h = new int64_t[np + 1];
        e = hipMemcpyAsync(h, a->ia0, sizeof(int64_t) * (np + 1), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e == hipSuccess)
            for (size_t i = 0; i <= np; ++i) ia[i] = (int)h[i] + 1;
        delete[] h;
    }
    if (e == hipSuccess && ja) e = hipMemcpyAsync(ja, a->ja, sizeof(int) * nz, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess && diag) e = hipMemcpyAsync(diag, a->diag, sizeof(int) * np, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess && mass) e = hipMemcpyAsync(mass, a->mass, sizeof(double) * nz, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess && lumped) e = hipMemcpyAsync(lumped, a->lumped, sizeof(double) * np, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess && cx) e = hipMemcpyAsync(cx, a->cx, sizeof(double) * nz, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess && cy) e = hipMemcpyAsync(cy, a->cy, sizeof(double) * nz, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return swe::fail(SWE_EHIP, "assembly read-back: %s", hipGetErrorString(e));
    return SWE_OK;
}

extern "C" int swe_assembly_destroy(swe_assembly* a) {
    release(a);
    return SWE_OK;
}

// =============================================================================================
// The sliced layout of an assembled mesh, built on the GPU (the same internal numbering and slots
// as build_layout on the host: rows stably sorted by length inside each tile's rows of the base order).
// =============================================================================================
namespace {

__global__ void k_lay_len(int np, const int64_t* __restrict__ ia0, int* __restrict__ lenc, int* __restrict__ bad) {
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= np) return;
    const int64_t l = ia0[i + 1] - ia0[i];
    lenc[i] = (int)l;
    if (l > swe::kMaxRow || l < 1) atomicOr(bad, 1);
}

// A set of rows in LDS, filled by a workgroup (open addressing; far past a halo's capacity it takes no more).
constexpr int kTileHash = 1024;
static_assert(kTileHash == 1024, "tile_hash gives 10 bits");
__device__ __forceinline__ int tile_hash(int j) { return (int)(((unsigned)j * 2654435761u) >> 22); }
__device__ __forceinline__ void tile_insert(int* key, int* count, int j) {
    for (int h = tile_hash(j), n = 0; n < kTileHash; ++n, h = (h + 1) & (kTileHash - 1)) {
        const int old = atomicCAS(key + h, -1, j);
        if (old == j) return;
        if (old == -1) {
            atomicAdd(count, 1);
            return;
        }
    }
}

// One workgroup per tile of the caller's numbering: sets *wide where its entries refer to more outside rows than a
// tile may have (which does not depend on the order of the rows within the tile).
__global__ void __launch_bounds__(256)
k_lay_fits(int np, int tile_slices, const int64_t* __restrict__ ia0, const int* __restrict__ ja, int* __restrict__ wide) {
    __shared__ int key[kTileHash];
    __shared__ int count;
    const int nsl = (np + 63) / 64, t0 = (int)blockIdx.x * tile_slices;
    const int ns = (nsl - t0 < tile_slices) ? nsl - t0 : tile_slices;
    const int row0 = t0 * 64, row1 = (row0 + 64 * ns < np) ? row0 + 64 * ns : np;
    for (int q = threadIdx.x; q < kTileHash; q += blockDim.x) key[q] = -1;
    if (threadIdx.x == 0) count = 0;
    __syncthreads();
    for (int r = row0 + (int)threadIdx.x; r < row1; r += blockDim.x)
        for (int64_t p = ia0[r]; p < ia0[r + 1]; ++p) {
            const int j = ja[p] - 1;
            if (j < row0 || j >= row1) tile_insert(key, &count, j);
        }
    __syncthreads();
    if (threadIdx.x == 0 && count > swe::tile_halo_cap(tile_slices, ns)) atomicOr(wide, 1);
}

// One workgroup per tile, one thread per row of it in the base order (base[p], or p when base is null): each
// row's rank among the tile's by (length, position in the base order); among its slice's where *wide is set.
__global__ void __launch_bounds__(64 * swe::kMaxTileSlices)
k_lay_sort(int np, const int* __restrict__ lenc, const int* __restrict__ base, const int* __restrict__ wide,
           int* __restrict__ perm) {
    __shared__ int key[64 * swe::kMaxTileSlices];
    const int n = (int)blockDim.x, k = (int)threadIdx.x;
    const int w0 = (int)blockIdx.x * n, pos = w0 + k;
    const int i = (pos < np) ? (base ? base[pos] : pos) : 0;
    const int mine = (pos < np) ? lenc[i] * n + k : 0x7fffffff;
    const int first = *wide ? (k & ~63) : 0, end = *wide ? first + 64 : n;
    key[k] = mine;
    __syncthreads();
    int rank = first;
    for (int m = first; m < end; ++m) rank += (key[m] < mine) ? 1 : 0;
    if (pos < np) perm[w0 + rank] = i;
}

// ---- locality order: nodes sorted along a Hilbert curve of their coordinates ------------------
// Orderable image of a double: unsigned comparison of the images orders finite doubles.
__device__ __forceinline__ unsigned long long ord_of(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
double double_of_ord(unsigned long long o) {
    const unsigned long long b = (o >> 63) ? (o & ~0x8000000000000000ull) : ~o;
    double v;
    std::memcpy(&v, &b, sizeof v);
    return v;
}

// box = {min x, max x, min y, max y} as orderable images (initialised to ~0, 0, ~0, 0).
__global__ void __launch_bounds__(256) k_bbox(int np, const double* __restrict__ rr, unsigned long long* __restrict__ box) {
    unsigned long long v[4] = {~0ull, 0ull, ~0ull, 0ull};
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < np; i += (int64_t)gridDim.x * blockDim.x) {
        const unsigned long long x = ord_of(rr[2 * i]), y = ord_of(rr[2 * i + 1]);
        v[0] = (x < v[0]) ? x : v[0];
        v[1] = (x > v[1]) ? x : v[1];
        v[2] = (y < v[2]) ? y : v[2];
        v[3] = (y > v[3]) ? y : v[3];
    }
    for (int off = 32; off > 0; off >>= 1)
        for (int q = 0; q < 4; ++q) {
            const unsigned long long o = __shfl_xor(v[q], off, 64);
            v[q] = (q & 1) ? ((o > v[q]) ? o : v[q]) : ((o < v[q]) ? o : v[q]);
        }
    // one atomic per workgroup and bound: they serialise on one cache line
    __shared__ unsigned long long red[4][4];
    const int w = (int)(threadIdx.x >> 6), q = (int)threadIdx.x;
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 4; ++k) red[k][w] = v[k];
    __syncthreads();
    if (q >= 4) return;
    unsigned long long r = red[q][0];
    for (int k = 1; k < 4; ++k) r = (q & 1) ? ((red[q][k] > r) ? red[q][k] : r) : ((red[q][k] < r) ? red[q][k] : r);
    if (q & 1) atomicMax(box + q, r);
    else atomicMin(box + q, r);
}

constexpr int kCurveBits = 20;   // per coordinate: 2^20 cells along each side of the bounding box

// Position of each node along a Hilbert curve through the 2^20 x 2^20 cells of the bounding box
// (the classic bit-by-bit conversion: quadrant, then rotate / reflect the lower bits).
__global__ void k_curve_key(int np, const double* __restrict__ rr, double x0, double sx, double y0, double sy,
                            unsigned long long* __restrict__ key, int* __restrict__ idx) {
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= np) return;
    const double top = (double)((1 << kCurveBits) - 1);
    double fx = (rr[2 * (size_t)i] - x0) * sx, fy = (rr[2 * (size_t)i + 1] - y0) * sy;
    fx = (fx > 0.0) ? ((fx < top) ? fx : top) : 0.0;
    fy = (fy > 0.0) ? ((fy < top) ? fy : top) : 0.0;
    unsigned x = (unsigned)fx, y = (unsigned)fy;
    unsigned long long d = 0;
    for (unsigned sq = 1u << (kCurveBits - 1); sq > 0; sq >>= 1) {
        const unsigned rx = (x & sq) ? 1u : 0u, ry = (y & sq) ? 1u : 0u;
        d += (unsigned long long)sq * sq * ((3u * rx) ^ ry);
        if (ry == 0) {
            if (rx == 1) {
                x = (x & ~(sq - 1)) + (sq - 1 - (x & (sq - 1)));
                y = (y & ~(sq - 1)) + (sq - 1 - (y & (sq - 1)));
            }
            const unsigned t = x;
            x = y;
            y = t;
        }
    }
    key[i] = d;
    idx[i] = i;
}

__global__ void k_lay_iperm(int np, int np_pad, const int* __restrict__ perm, const int* __restrict__ lenc,
                            int* __restrict__ iperm, int* __restrict__ lenr) {
    const int r = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (r >= np_pad) return;
    if (r < np) {
        const int i = perm[r];
        iperm[i] = r;
        lenr[r] = lenc[i];
    } else {
        lenr[r] = 0;
    }
}

// Per slice: 64 x its longest row (slots) and its off-diagonal entries (compact-list length).
__global__ void k_lay_slices(int nsl, int np, const int* __restrict__ lenr, int64_t* __restrict__ slots,
                             int64_t* __restrict__ ecnt, int* __restrict__ wmax) {
    const int s = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (s == nsl) slots[s] = ecnt[s] = 0;
    if (s >= nsl) return;
    int w = 0;
    int64_t e = 0;
    for (int l = 0; l < 64; ++l) {
        const int r = s * 64 + l;
        const int L = lenr[r];
        w = (L > w) ? L : w;
        if (r < np) e += L - 1;
    }
    slots[s] = 64 * (int64_t)w;
    ecnt[s] = e;
    atomicMax(wmax, w);
}

// What the host reads of a layout: its slots, its list entries, the row-length check and the longest row.
__global__ void k_lay_sums(int nsl, const int64_t* __restrict__ sptr, const int64_t* __restrict__ eoff,
                           const int* __restrict__ flag, int64_t* __restrict__ sums) {
    if (threadIdx.x != 0) return;
    sums[0] = sptr[nsl];
    sums[1] = eoff[nsl];
    sums[2] = flag[0];
    sums[3] = flag[1];
}

struct LayOut {
    uint8_t* len8;
    uint8_t* dpos8;
    uint8_t* dirm;
    int* perm;
    double* m;
    double* z;
    int* col;
    int16_t* dcol;
    double2* c;
};

// Per internal row: its slots (columns, offsets, c_ij) and node data, as build_layout fills them.
__global__ void k_lay_fill(int np, int np_pad, int64_t r0, int64_t p0, const int* __restrict__ perm,
                           const int* __restrict__ iperm, const int* __restrict__ lenr,
                           const int64_t* __restrict__ sptr, const int64_t* __restrict__ ia0,
                           const int* __restrict__ ja, const double* __restrict__ cx, const double* __restrict__ cy,
                           const double* __restrict__ lumped, const double* __restrict__ bath, LayOut o,
                           int64_t* __restrict__ csr2slot) {
    const int r = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (r >= np_pad) return;
    o.dirm[r0 + r] = 0;
    if (r >= np) {
        o.len8[r0 + r] = 0;
        o.dpos8[r0 + r] = 0;
        return;
    }
    const int i = perm[r];
    const int L = lenr[r];
    const int64_t base = sptr[r >> 6] + (r & 63);
    const int64_t pi = ia0[i];
    int dp = 0;
    for (int q = 0; q < L; ++q) {
        const int64_t p = pi + q;
        const int j = ja[p] - 1;
        const int jr = iperm[j];
        const int64_t slot = base + 64 * (int64_t)q;
        o.col[p0 + slot] = (int)(r0 + jr);
        const int off = jr - r;
        o.dcol[p0 + slot] = (int16_t)((off > swe::kColFar && off <= 32767) ? off : swe::kColFar);
        o.c[p0 + slot] = make_double2(cx[p], cy[p]);
        if (csr2slot) csr2slot[p] = slot;
        if (j == i) dp = q;
    }
    o.len8[r0 + r] = (uint8_t)L;
    o.dpos8[r0 + r] = (uint8_t)dp;
    o.perm[r0 + r] = i;
    o.m[r0 + r] = lumped[i];
    o.z[r0 + r] = bath[i];
}

// One wave per slice: its compact list of off-diagonal slots, entry by entry, lanes in order.
__global__ void k_lay_elist(int nsl, int np, int64_t r0, int64_t e0, const int* __restrict__ lenr,
                            const uint8_t* __restrict__ dpos8, const int64_t* __restrict__ sptr,
                            const int64_t* __restrict__ eoff, uint16_t* __restrict__ elist) {
    const int s = (int)(blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6));
    if (s >= nsl) return;
    const int lane = (int)(threadIdx.x & 63);
    const int r = s * 64 + lane;
    const int L = (r < np) ? lenr[r] : 0;
    const int dp = (r < np) ? (int)dpos8[r0 + r] : 0;
    const int w = (int)((sptr[s + 1] - sptr[s]) / 64);
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int64_t off = eoff[s];
    for (int q = 0; q < w; ++q) {
        const bool active = q < L && q != dp;
        const unsigned long long mask = __ballot(active);
        if (active) elist[e0 + off + __popcll(mask & below)] = (uint16_t)(q * 64 + lane);
        off += __popcll(mask);
    }
}

__global__ void k_lay_slice_info(int nsl, int64_t s0, int64_t p0, int64_t e0, int inst, int tile_slices,
                                 const int64_t* __restrict__ sptr, const int64_t* __restrict__ eoff,
                                 swe::SliceInfo* __restrict__ sl) {
    const int s = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (s >= nsl) return;
    swe::SliceInfo v;
    v.sbase = p0 + sptr[s];
    v.ebase = e0 + eoff[s];
    v.inst = inst;
    v.ecount = (int)(eoff[s + 1] - eoff[s]);
    v.tile_slices = (s % tile_slices) ? 0 : ((nsl - s < tile_slices) ? nsl - s : tile_slices);
    v.nhalo = 0;
    sl[s0 + s] = v;
}

// One workgroup per tile: the distinct rows outside the tile that its entries refer to, collected in a hash
// set in LDS (a tile past the halo capacity gives up),
// ranked by counting (ascending, as the host layout sorts them), every entry's column within the tile,
// and the longest list (INT_MAX: one past the capacity).  Runs after k_lay_fill (global columns) and k_lay_slice_info.
__global__ void __launch_bounds__(256)
k_lay_tiles(int nsl, int64_t s0, int tile_slices, const uint8_t* __restrict__ len8, const int* __restrict__ col,
            swe::SliceInfo* __restrict__ sl, uint16_t* __restrict__ lcol, int* __restrict__ halo,
            int* __restrict__ longest) {
    __shared__ int key[kTileHash];
    __shared__ int pos[kTileHash];
    __shared__ int list[512];
    __shared__ int count;
    const int t0 = (int)blockIdx.x * tile_slices;
    const int ns = (nsl - t0 < tile_slices) ? nsl - t0 : tile_slices;
    const int64_t g0 = s0 + t0;                       // the tile's first slice
    const int row0 = (int)(g0 * 64), row1 = row0 + 64 * ns;
    const int cap = swe::tile_halo_cap(tile_slices, ns);
    for (int q = threadIdx.x; q < kTileHash; q += blockDim.x) key[q] = -1;
    if (threadIdx.x == 0) count = 0;
    __syncthreads();
    for (int r = threadIdx.x; r < 64 * ns; r += blockDim.x) {
        const int L = len8[row0 + r];
        const int64_t base = sl[g0 + (r >> 6)].sbase + (r & 63);
        for (int q = 0; q < L; ++q) {
            const int j = col[base + 64 * (int64_t)q];
            if (j >= row0 && j < row1) continue;
            tile_insert(key, &count, j);
        }
    }
    __syncthreads();
    const int n = count;
    if (threadIdx.x == 0) atomicMax(longest, (n > cap) ? 0x7fffffff : n);
    if (n > cap) return;
    __syncthreads();
    if (threadIdx.x == 0) count = 0;
    __syncthreads();
    for (int h = threadIdx.x; h < kTileHash; h += blockDim.x)
        if (key[h] >= 0) list[atomicAdd(&count, 1)] = key[h];
    __syncthreads();
    for (int h = threadIdx.x; h < kTileHash; h += blockDim.x) {
        const int k = key[h];
        if (k < 0) continue;
        int rank = 0;
        for (int q = 0; q < n; ++q) rank += (list[q] < k) ? 1 : 0;
        pos[h] = rank;
        halo[g0 * swe::kHaloStride + rank] = k;
    }
    if (threadIdx.x == 0) sl[g0].nhalo = n;
    __syncthreads();
    for (int r = threadIdx.x; r < 64 * ns; r += blockDim.x) {
        const int L = len8[row0 + r];
        const int64_t base = sl[g0 + (r >> 6)].sbase + (r & 63);
        for (int q = 0; q < L; ++q) {
            const int64_t p = base + 64 * (int64_t)q;
            const int j = col[p];
            int l = j - row0;
            if (j < row0 || j >= row1) {
                int h = tile_hash(j);
                while (key[h] != j) h = (h + 1) & (kTileHash - 1);
                l = 64 * tile_slices + pos[h];
            }
            lcol[p] = (uint16_t)l;
        }
    }
}

__global__ void k_lay_bc(int nbc, int nh, int nux, int64_t r0, int64_t b0, int inst, const int* __restrict__ nodes1,
                         const int* __restrict__ iperm, swe::BcEntry* __restrict__ bc, uint8_t* __restrict__ dirm) {
    const int q = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (q >= nbc) return;
    const int comp = (q < nh) ? 0 : (q < nh + nux) ? 1 : 2;
    const int row = (int)(r0 + iperm[nodes1[q] - 1]);
    bc[b0 + q] = swe::BcEntry{row, inst, comp, (int)(b0 + q)};
    // several entries may share a row and rows share a word: set the row's bit in its aligned word
    atomicOr((unsigned*)dirm + (row >> 2), 1u << (8 * (row & 3) + comp));
}

}  // namespace

namespace {

hipError_t read_u64(const unsigned long long* d, unsigned long long* h, int n, hipStream_t s) {
    hipError_t e = hipMemcpyAsync(h, d, sizeof(unsigned long long) * (size_t)n, hipMemcpyDeviceToHost, s);
    return (e == hipSuccess) ? hipStreamSynchronize(s) : e;
}

// Scratch of the locality order.
struct OrderWork {
    unsigned long long *box = nullptr, *keys = nullptr, *keys2 = nullptr;
    int *idx = nullptr, *order = nullptr;
    char* tmp = nullptr;
    size_t bytes = 0;
    bool used = false;
    void add(swe::Carver& c, int np) {
        used = swe::reorder_enabled() && np >= 2;
        if (!used) return;
        (void)hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, keys, keys2, idx, order, np, 0, 2 * kCurveBits, nullptr);
        c.add(&box, 4);
        c.add(&keys, (size_t)np);
        c.add(&keys2, (size_t)np);
        c.add(&idx, (size_t)np);
        c.add(&order, (size_t)np);
        c.add(&tmp, bytes);
    }
};

// The base order of the layout: the nodes along a Hilbert curve of their coordinates, the device
// counterpart of the host layout's locality order, or the caller's numbering (*base null) under
// SWE_REORDER=0.  Only the processing order changes; results do not depend on it.
hipError_t locality_order(const swe_assembly* a, hipStream_t s, OrderWork& w, const int** base) {
    *base = nullptr;
    const int np = a->np;
    if (!w.used) return hipSuccess;
    unsigned long long h[4] = {~0ull, 0ull, ~0ull, 0ull};
    const unsigned bl = grid_of(np, 256);
    hipError_t e = hipMemcpyAsync(w.box, h, sizeof h, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_bbox, dim3(bl < 256u ? bl : 256u), dim3(256), 0, s, np, (const double*)a->rr, w.box);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = read_u64(w.box, h, 4, s);
    if (e != hipSuccess) return e;
    const double x0 = double_of_ord(h[0]), x1 = double_of_ord(h[1]);
    const double y0 = double_of_ord(h[2]), y1 = double_of_ord(h[3]);
    const double top = (double)((1 << kCurveBits) - 1);
    const double sx = (x1 > x0) ? top / (x1 - x0) : 0.0, sy = (y1 > y0) ? top / (y1 - y0) : 0.0;
    hipLaunchKernelGGL(k_curve_key, dim3(bl), dim3(256), 0, s, np, (const double*)a->rr, x0, sx, y0, sy, w.keys, w.idx);
    // a radix sort is stable: equal keys keep the caller's order
    e = hipcub::DeviceRadixSort::SortPairs(w.tmp, w.bytes, w.keys, w.keys2, w.idx, w.order, np, 0, 2 * kCurveBits, s);
    if (e == hipSuccess) *base = w.order;
    return e;
}

}  // namespace

namespace swe {

void free_device_layout(DeviceLayout& DL) {
    dfree(DL.block, DL.stream);
    DL = DeviceLayout{};
}

int64_t assembly_rows(const swe_assembly* a) { return ((int64_t)a->np + 63) / 64 * 64; }

int build_layout_device(const swe_assembly* a, int tile_slices, DeviceLayout& DL) {
    if (!a) return fail(SWE_EINVAL, "null assembly");
    DL = DeviceLayout{};
    const int np = a->np;
    DL.np = np;
    DL.nnz = a->nnz;
    const int nsl = (np + 63) / 64, np_pad = nsl * 64;
    DL.nsl = nsl;
    hipStream_t s = a->stream;
    DL.stream = s;
    int* lenc = nullptr;
    int* flag = nullptr;
    int64_t *slots = nullptr, *ecnt = nullptr;
    int64_t* sums = nullptr;
    char* tmp = nullptr;
    void* work = nullptr;
    const size_t nscan = scan_bytes(nsl + 1);
    Carver keep, temp;
    keep.add(&DL.perm, (size_t)np);
    keep.add(&DL.iperm, (size_t)np);
    keep.add(&DL.len, (size_t)np_pad);
    keep.add(&DL.sptr, (size_t)nsl + 1);
    keep.add(&DL.eoff, (size_t)nsl + 1);
    temp.add(&flag, 3);        // row-length check, longest row, halos too long
    const size_t zeroed = temp.bytes();
    temp.add(&sums, 4);
    temp.add(&lenc, (size_t)np);
    temp.add(&slots, (size_t)nsl + 1);
    temp.add(&ecnt, (size_t)nsl + 1);
    temp.add(&tmp, nscan);
    OrderWork ow;
    ow.add(temp, np);
    hipError_t e = block_alloc(keep, &DL.block, s);
    if (e == hipSuccess) e = block_alloc(temp, &work, s);
    if (e == hipSuccess) e = hipMemsetAsync(work, 0, zeroed, s);
    const int* base = nullptr;
    if (e == hipSuccess) e = locality_order(a, s, ow, &base);
    int64_t h[4] = {0, 0, 0, 0};
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_lay_len, dim3(grid_of(np, 256)), dim3(256), 0, s, np, (const int64_t*)a->ia0, lenc, flag);
        // a numbering of the caller's may be no order for tiles (build_layout says why the windows are slices there)
        if (!base && tile_slices > 1)
            hipLaunchKernelGGL(k_lay_fits, dim3(grid_of(nsl, tile_slices)), dim3(256), 0, s, np, tile_slices,
                               (const int64_t*)a->ia0, (const int*)a->ja, flag + 2);
        hipLaunchKernelGGL(k_lay_sort, dim3(grid_of(nsl, tile_slices)), dim3(64 * tile_slices), 0, s, np,
                           (const int*)lenc, base, (const int*)(flag + 2), DL.perm);
        hipLaunchKernelGGL(k_lay_iperm, dim3(grid_of(np_pad, 256)), dim3(256), 0, s, np, np_pad, (const int*)DL.perm,
                           (const int*)lenc, DL.iperm, DL.len);
        hipLaunchKernelGGL(k_lay_slices, dim3(grid_of(nsl + 1, 256)), dim3(256), 0, s, nsl, np, (const int*)DL.len, slots,
                           ecnt, flag + 1);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = exclusive_scan(slots, DL.sptr, nsl + 1, tmp, nscan, s);
    if (e == hipSuccess) e = exclusive_scan(ecnt, DL.eoff, nsl + 1, tmp, nscan, s);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_lay_sums, dim3(1), dim3(64), 0, s, nsl, (const int64_t*)DL.sptr, (const int64_t*)DL.eoff,
                           (const int*)flag, sums);
        e = hipMemcpyAsync(h, sums, sizeof h, hipMemcpyDeviceToHost, s);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    dfree(work, s);
    if (e != hipSuccess) {
        free_device_layout(DL);
        return fail(SWE_EHIP, "device layout: %s", hipGetErrorString(e));
    }
    if (h[2]) {
        free_device_layout(DL);
        return fail(SWE_EINVAL, "a row has more than %d entries", kMaxRow);
    }
    DL.nslot = h[0];
    DL.ne = h[1];
    DL.wmax = (int)h[3];
    return SWE_OK;
}

int pool_add_assembled(Pool* P, const swe_assembly* a, const DeviceLayout& DL, const double* bath,
                       const int* const lists[3], const int nlist[3], const swe_params& prm, const double* un,
                       double t0, double tfinal, long long max_steps, int* id, int64_t* csr2slot) {
    if (!a || !bath || !id) return fail(SWE_EINVAL, "null argument");
    Mode md;
    int rc = mode_of(prm, md);
    if (rc) return rc;
    if (P->mode_set && !same_mode(md, P->mode)) return fail(SWE_EBADOPT, "this instance's scheme differs from the pool's");
    if ((rc = check_sgn_lists(md, nlist[1], nlist[2]))) return rc;
    if (md.sgn && (rc = ensure_sgn_buffers(P))) return rc;
    const int np = DL.np;
    for (int c = 0; c < 3; ++c) {
        if (nlist[c] < 0 || (nlist[c] > 0 && !lists[c])) return fail(SWE_EINVAL, "Dirichlet list %d is malformed", c);
        for (int q = 0; q < nlist[c]; ++q)
            if (lists[c][q] < 1 || lists[c][q] > np) return fail(SWE_EINVAL, "Dirichlet node %d out of range", lists[c][q]);
    }
    int k = -1;
    for (int q = 0; q < P->inst_cap; ++q)
        if (!P->inst[(size_t)q].used) { k = q; break; }
    const int64_t nbc = (int64_t)nlist[0] + nlist[1] + nlist[2];
    const int64_t s0 = (k < 0) ? -1 : P->a_slices.alloc(DL.nsl);
    const int64_t p0 = (s0 < 0) ? -1 : P->a_slots.alloc(DL.nslot);
    const int64_t e0 = (p0 < 0) ? -1 : P->a_elist.alloc(DL.ne);
    const int64_t b0 = (e0 < 0) ? -1 : P->a_bc.alloc(nbc);
    if (k < 0 || s0 < 0 || p0 < 0 || e0 < 0 || b0 < 0) {
        if (s0 >= 0) P->a_slices.release(s0, DL.nsl);
        if (p0 >= 0) P->a_slots.release(p0, DL.nslot);
        if (e0 >= 0) P->a_elist.release(e0, DL.ne);
        return fail(SWE_EFULL, "the pool has no room for a mesh of %d nodes now", np);
    }
    const int64_t r0 = s0 * 64;
    const int np_pad = DL.nsl * 64;
    // the admission runs on the pool's copy stream, as an upload does: the steps queued on the compute
    // stream go on meanwhile (the new rows are not in their launch lists yet)
    hipStream_t s = P->copy;
    double* dbath = nullptr;
    int* dnodes = nullptr;
    int* dlong = nullptr;
    int longest = 0;
    void* work = nullptr;
    Carver temp;
    temp.add(&dlong, 1);
    temp.add(&dbath, (size_t)np);
    temp.add(&dnodes, (size_t)nbc);
    hipError_t e = block_alloc(temp, &work, s);
    if (e == hipSuccess) e = hipMemcpyAsync(dlong, &longest, sizeof longest, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemcpyAsync(dbath, bath, sizeof(double) * (size_t)np, hipMemcpyHostToDevice, s);
    for (int c = 0, q = 0; c < 3 && e == hipSuccess; q += nlist[c], ++c)
        if (nlist[c] > 0)
            e = hipMemcpyAsync(dnodes + q, lists[c], sizeof(int) * (size_t)nlist[c], hipMemcpyHostToDevice, s);
    // ranges freed by a removal are rewritten only after the removal's kernels
    if (e == hipSuccess) e = hipStreamWaitEvent(s, P->released, 0);
    if (e == hipSuccess && un) {
        const int nc = md.sgn ? 5 : 3;
        double* st = md.sgn ? P->stage5 : P->stage3;
        e = hipMemcpyAsync(st + nc * r0, un, sizeof(double) * nc * (size_t)np, hipMemcpyHostToDevice, s);
    }
    if (e == hipSuccess) {
        LayOut o{P->len, P->dpos, P->dirm, P->perm, P->m, P->z, P->col, P->dcol, P->c};
        hipLaunchKernelGGL(k_lay_fill, dim3(grid_of(np_pad, 256)), dim3(256), 0, s, np, np_pad, r0, p0,
                           (const int*)DL.perm, (const int*)DL.iperm, (const int*)DL.len, (const int64_t*)DL.sptr,
                           (const int64_t*)a->ia0, (const int*)a->ja, (const double*)a->cx, (const double*)a->cy,
                           (const double*)a->lumped, (const double*)dbath, o, csr2slot);
        hipLaunchKernelGGL(k_lay_elist, dim3(grid_of(DL.nsl, 4)), dim3(256), 0, s, DL.nsl, np, r0, e0,
                           (const int*)DL.len, (const uint8_t*)P->dpos, (const int64_t*)DL.sptr,
                           (const int64_t*)DL.eoff, P->elist);
        hipLaunchKernelGGL(k_lay_slice_info, dim3(grid_of(DL.nsl, 256)), dim3(256), 0, s, DL.nsl, s0, p0, e0, k,
                           P->tile_slices, (const int64_t*)DL.sptr, (const int64_t*)DL.eoff, P->sl);
        hipLaunchKernelGGL(k_lay_tiles, dim3(grid_of(DL.nsl, P->tile_slices)), dim3(256), 0, s, DL.nsl, s0,
                           P->tile_slices, (const uint8_t*)P->len, (const int*)P->col, P->sl, P->lcol, P->halo, dlong);
        if (nbc > 0)
            hipLaunchKernelGGL(k_lay_bc, dim3(grid_of(nbc, 256)), dim3(256), 0, s, (int)nbc, nlist[0], nlist[1], r0, b0,
                               k, (const int*)dnodes, (const int*)DL.iperm, P->bc, P->dirm);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&longest, dlong, sizeof longest, hipMemcpyDeviceToHost, s);
    dfree(work, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        P->a_slices.release(s0, DL.nsl);
        P->a_slots.release(p0, DL.nslot);
        P->a_elist.release(e0, DL.ne);
        P->a_bc.release(b0, nbc);
        return fail(SWE_EHIP, "admission of an assembled mesh: %s", hipGetErrorString(e));
    }
    InstHost I;
    I.np = np;
    I.nnz = (int)DL.nnz;
    I.np_pad = np_pad;
    I.wmax = DL.wmax;
    I.slice0 = s0;
    I.nslices = DL.nsl;
    I.slot0 = p0;
    I.nslots = DL.nslot;
    I.e0 = e0;
    I.ne = DL.ne;
    I.bc0 = b0;
    I.nbc = nbc;
    I.nh = nlist[0];
    I.nux = nlist[1];
    I.nuy = nlist[2];
    I.max_halo = (longest == 0x7fffffff) ? -1 : longest;
    if ((rc = pool_activate(P, k, I, prm, un != nullptr, t0, tfinal, max_steps))) return rc;
    *id = k;
    return SWE_OK;
}

}  // namespace swe
