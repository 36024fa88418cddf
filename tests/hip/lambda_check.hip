// lambda_check.hip -- TEST INFRASTRUCTURE: the library's wave speed and shared divisions on the GPU.
//
//   lambda_check IN OUT    IN: doubles gravity, htiny, then records (hl, qxl, qyl, hr, qxr, qyr, n1, n2);
//                          OUT: swe::lambda_vacc of each record
//   lambda_check COUNT     swe::div_shared against the division, bit for bit (zeros of either sign
//                          equal), on 2^COUNT hashed operand pairs of each class; exits with 3 when any differs
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "swe_kernels.h"

namespace {

__global__ void k_lambda(int n, const double* __restrict__ rec, swe::Consts K, double* __restrict__ out) {
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n) return;
    const double* r = rec + 8 * (size_t)i;
    int err = 0;
    out[i] = swe::lambda_vacc(r[0], r[1], r[2], r[3], r[4], r[5], r[6], r[7], swe::ovh_of(r[0], K.htiny),
                              swe::ovh_of(r[3], K.htiny), sqrt(K.g * fabs(r[0])), sqrt(K.g * fabs(r[3])), K,
                              swe::uniform_rcp(K.g16), err);
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
__device__ __forceinline__ double make(uint64_t sign, uint64_t e, uint64_t man) {
    return __longlong_as_double((long long)((sign << 63) | (e << 52) | (man & 0xfffffffffffffull)));
}

// class 0: both in [2^-20, 2^20]; 1: mantissas near all zeros or ones; 2: exponents across the ranges the
// shared form covers and past them; 3: any bit patterns; 4: zeros, infinities, denormals as dividend
__global__ void k_div(uint64_t n, uint64_t seed, int cls, unsigned long long* bad, double* ex) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    unsigned long long nb = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint64_t r = mix64(i ^ seed), s = mix64(r);
        double a, b;
        if (cls == 0) {
            a = make(r >> 63, 1003 + (r >> 52) % 41, r);
            b = make(0, 1003 + (s >> 52) % 41, s);
        } else if (cls == 1) {
            a = make(r >> 63, 1003 + (r >> 52) % 41, (r & 1) ? 0xfffffffffffffull - (r >> 1 & 0xff) : (r >> 1 & 0xff));
            b = make(0, 1003 + (s >> 52) % 41, (s & 1) ? 0xfffffffffffffull - (s >> 1 & 0xff) : (s >> 1 & 0xff));
        } else if (cls == 2) {
            a = make(r >> 63, 500 + (r >> 52) % 1047, r);
            b = make(0, 700 + (s >> 52) % 647, s);
        } else if (cls == 3) {
            a = __longlong_as_double((long long)r);
            b = __longlong_as_double((long long)s);
        } else {
            a = (r & 3) == 0 ? 0.0 : (r & 3) == 1 ? make(0, 2047, 0) : (r & 3) == 2 ? make(0, 0, r) : make(0, (r >> 52) % 600, r);
            b = make(0, 923 + (s >> 52) % 201, s);
        }
        const double q = a / b, p = swe::div_shared(a, swe::refined_rcp(b));
        const bool same = __double_as_longlong(p) == __double_as_longlong(q) || (p == 0.0 && q == 0.0) || (p != p && q != q);
        if (!same) {
            ++nb;
            ex[0] = a;
            ex[1] = b;
        }
    }
    if (nb) atomicAdd(bad, nb);
}

int check_div(int lg) {
    unsigned long long* bad = nullptr;
    double* ex = nullptr;
    if (hipMalloc((void**)&bad, sizeof *bad) != hipSuccess || hipMalloc((void**)&ex, 2 * sizeof *ex) != hipSuccess) return 1;
    int rc = 0;
    for (int cls = 0; cls < 5; ++cls) {
        unsigned long long h = 0;
        double e[2] = {0.0, 0.0};
        if (hipMemset(bad, 0, sizeof *bad) != hipSuccess) return 1;
        hipLaunchKernelGGL(k_div, dim3(8192), dim3(256), 0, 0, 1ull << lg, 0xd1f0000ull + (uint64_t)cls, cls, bad, ex);
        if (hipMemcpy(&h, bad, sizeof h, hipMemcpyDeviceToHost) != hipSuccess) return 1;
        if (h && hipMemcpy(e, ex, sizeof e, hipMemcpyDeviceToHost) != hipSuccess) return 1;
        std::printf("class %d: %llu of %llu differ", cls, h, 1ull << lg);
        if (h) {
            std::printf(" (for instance %.17g / %.17g)", e[0], e[1]);
            rc = 3;
        }
        std::printf("\n");
    }
    (void)hipFree(bad);
    (void)hipFree(ex);
    return rc;
}

}  // namespace

int main(int argc, char** argv) {
    if (argc == 2) {
        const int lg = std::atoi(argv[1]);
        if (lg < 10 || lg > 32) return 2;
        return check_div(lg);
    }
    if (argc != 3) return 2;
    FILE* f = std::fopen(argv[1], "rb");
    if (!f) return 2;
    double head[2];
    if (std::fread(head, sizeof(double), 2, f) != 2) return 2;
    std::vector<double> rec;
    double buf[8];
    while (std::fread(buf, sizeof(double), 8, f) == 8) rec.insert(rec.end(), buf, buf + 8);
    std::fclose(f);
    const int n = (int)(rec.size() / 8);
    if (n == 0) return 2;
    swe::Consts K{};
    const double g = head[0], t = 2.0 * std::sqrt(2.0) - 1.0;
    K.g = g;
    K.htiny = head[1];
    K.x0 = t * t;
    K.a_c2 = 1 / (2.0 * std::sqrt(2.0));
    K.two_sqrt_g = 2 * std::sqrt(g);
    K.sqrt_2_g = std::sqrt(2 / g);
    K.g_half = g / 2;
    K.g16 = 16 * g;
    K.lam_w = 1.01 / (2.34 * 2.34 * K.g_half);
    K.lam_h = 0x1p+300;
    double *dr = nullptr, *dout = nullptr;
    std::vector<double> out((size_t)n);
    if (hipMalloc((void**)&dr, sizeof(double) * rec.size()) != hipSuccess) return 1;
    if (hipMalloc((void**)&dout, sizeof(double) * out.size()) != hipSuccess) return 1;
    if (hipMemcpy(dr, rec.data(), sizeof(double) * rec.size(), hipMemcpyHostToDevice) != hipSuccess) return 1;
    hipLaunchKernelGGL(k_lambda, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, n, dr, K, dout);
    if (hipMemcpy(out.data(), dout, sizeof(double) * out.size(), hipMemcpyDeviceToHost) != hipSuccess) return 1;
    (void)hipFree(dr);
    (void)hipFree(dout);
    f = std::fopen(argv[2], "wb");
    if (!f || std::fwrite(out.data(), sizeof(double), out.size(), f) != out.size()) return 2;
    return std::fclose(f) ? 2 : 0;
}
