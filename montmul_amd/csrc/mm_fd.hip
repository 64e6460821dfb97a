// mm_fd.hip - the double-precision step kernels of every length they run (L = 2,048 .. 32,768), in an
// object of their own, and their tables.

#include "mm_fd.h"

#include <algorithm>
#include <cmath>

namespace mm {
namespace fd {

// Four waves per SIMD (128 VGPRs): two 512-thread workgroups, or one of 1,024, on a CU.
template <u32 LOGC, bool BARE>
__global__ __launch_bounds__(Geo<LOGC>::T) __attribute__((amdgpu_waves_per_eu(4))) void k_steps_fd(Args A, u32 bits) {
    extern __shared__ __align__(16) unsigned char lds[];
    steps<LOGC, BARE>(A, blockIdx.x, bits, lds);
}

template <u32 LOGC>
__global__ __launch_bounds__(Geo<LOGC>::T) __attribute__((amdgpu_waves_per_eu(4))) void k_constants_fd(Args A, const u32* npl, const u32* nl,
                                                                                                  double2* np, double2* nh) {
    extern __shared__ __align__(16) unsigned char lds[];
    typedef Slot<LOGC> S;
    const size_t v = blockIdx.x;
    constants<LOGC>(A, npl + v * S::k, nl + v * S::k, np + v * S::C, nh + v * S::H, lds);
}

template <bool BARE> __global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4))) void k_steps_fd_split(Args A, u32 bits) {
    extern __shared__ __align__(16) unsigned char lds[];
    steps_split<BARE>(A, blockIdx.x, bits, lds);
}
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4))) void k_constants_fd_split(Args A, const u32* npl, const u32* nl, double2* np,
                                                                                                double2* nh, u32* dig) {
    extern __shared__ __align__(16) unsigned char lds[];
    typedef SplitSlot S;
    const size_t v = blockIdx.x;
    constants_split(A, npl + v * S::K, nl + v * S::K, np + v * 2 * S::H, nh + v * S::H, dig + v * S::H, lds);
}

// One product; four waves per SIMD as the steps, whose code it shares.
template <u32 LOGC>
__global__ __launch_bounds__(LOGC == 15 ? 1024 : Geo<LOGC == 15 ? 14 : LOGC>::T) __attribute__((amdgpu_waves_per_eu(4))) void k_mul_fd(
    Args A, u32 out, u32 a, u32 b, double2* spec) {
    extern __shared__ __align__(16) unsigned char lds[];
    if constexpr (LOGC == 15)
        product_split(A, out, a, b, spec, lds);
    else
        product<LOGC>(A, out, a, b, spec, lds);
}

template <u32 LOGC>
__global__ __launch_bounds__(LOGC == 15 ? 1024 : Geo<LOGC == 15 ? 14 : LOGC>::T) __attribute__((amdgpu_waves_per_eu(4))) void k_plain_fd(
    Args A, u32 first, u32* out, u32* T) {
    extern __shared__ __align__(16) unsigned char lds[];
    constexpr size_t k = 1u << (LOGC - 1);
    const size_t row = blockIdx.x;
    if constexpr (LOGC == 15)
        plain_split(A, first + blockIdx.x, out + row * k, T + row * 2 * k, lds);
    else
        plain<LOGC>(A, first + blockIdx.x, out + row * k, T + row * 2 * k, lds);
}

// k = 1,024 .. 16,384 limbs; c C < 2^17 keeps the limb sums of T below BETA (2^32 - 1) (sums_fit).
bool fits(u32 k, u32 base) { return k >= 1024 && k <= 16384 && (k & (k - 1)) == 0 && (u64)base * 2 * k < 131072; }

double2 unit(u64 num, u64 den) {
    // The octant's sine and cosine, so that both are rounded from small angles.
    num %= den;
    const u64 q = num / (den / 4), r = num % (den / 4);
    const bool flip = r > den / 8;
    const long double a = 2 * 3.14159265358979323846264338327950288L * (long double)(flip ? den / 4 - r : r) / (long double)den;
    double c = (double)cosl(a), s = (double)sinl(a);
    if (flip) std::swap(c, s);
    switch (q) {
        case 0: return make_double2(c, s);
        case 1: return make_double2(-s, c);
        case 2: return make_double2(-c, -s);
        default: return make_double2(s, -c);
    }
}

void make_tables(u32 C, double2* out) {
    const u32 T = C / 16, S1 = C / 256, S2 = C / 4096;
    for (u32 a = 0; a < 4; a++)
        for (u32 t = 0; t < T; t++) out[a * T + t] = unit((u64)t * (16 * a + 1), 4ull * C);
    for (u32 b = 1; b < 4; b++)
        for (u32 t = 0; t < T; t++) out[(3 + b) * T + t] = unit((u64)t * b, C);
    out += 7 * T;
    for (u32 m = 0; m < 16; m++)
        for (u32 j = 0; j < S1; j++) out[m * S1 + j] = unit((u64)j * m, T);
    out += C / 16;
    for (u32 m = 0; m < 16; m++)
        for (u32 j = 0; j < S2; j++) out[m * S2 + j] = unit((u64)j * m, S1);
    out += C / 256;
    for (u32 p = 0; p < 2; p++)
        for (u32 a = 0; a < 4; a++)
            for (u32 t = 0; t < T; t++) out[(4 * p + a) * T + t] = unit((u64)t * (32 * a + 4 * p + 1), 8ull * C);
    for (u32 p = 0; p < 2; p++)
        for (u32 e = 0; e < 16; e++) out[8 * T + 16 * p + e] = unit((4ull * p + 1) * e, 128);
}

template <u32 LOGC> static hipError_t limit() {
    for (const void* k : {(const void*)k_steps_fd<LOGC, false>, (const void*)k_steps_fd<LOGC, true>, (const void*)k_constants_fd<LOGC>,
                          (const void*)k_mul_fd<LOGC>, (const void*)k_plain_fd<LOGC>}) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Geo<LOGC>::lds);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
hipError_t set_lds_limit() {
    hipError_t e = limit<11>();
    if (e == hipSuccess) e = limit<12>();
    if (e == hipSuccess) e = limit<13>();
    if (e == hipSuccess) e = limit<14>();
    for (const void* k : {(const void*)k_steps_fd_split<false>, (const void*)k_steps_fd_split<true>, (const void*)k_constants_fd_split, (const void*)k_mul_fd<15>,
                          (const void*)k_plain_fd<15>})
        if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Geo<14>::lds);
    return e;
}

template <u32 LOGC> static hipError_t go(const Args& A, u32 slots, u32 bits, bool bare, hipStream_t sm) {
    typedef Geo<LOGC> G;
    if (bare)
        hipLaunchKernelGGL((k_steps_fd<LOGC, true>), dim3(slots), dim3(G::T), G::lds, sm, A, bits);
    else
        hipLaunchKernelGGL((k_steps_fd<LOGC, false>), dim3(slots), dim3(G::T), G::lds, sm, A, bits);
    return hipGetLastError();
}
hipError_t launch(const Args& A, u32 k, u32 slots, u32 bits, bool bare, hipStream_t sm) {
    switch (k) {
        case 1024: return go<11>(A, slots, bits, bare, sm);
        case 2048: return go<12>(A, slots, bits, bare, sm);
        case 4096: return go<13>(A, slots, bits, bare, sm);
        case 8192: return go<14>(A, slots, bits, bare, sm);
        case 16384:
            if (bare)
                hipLaunchKernelGGL((k_steps_fd_split<true>), dim3(slots), dim3(1024), Geo<14>::lds, sm, A, bits);
            else
                hipLaunchKernelGGL((k_steps_fd_split<false>), dim3(slots), dim3(1024), Geo<14>::lds, sm, A, bits);
            return hipGetLastError();
        default: return hipErrorInvalidValue;
    }
}

template <u32 LOGC>
static hipError_t consts(const Args& A, u32 count, const u32* npl, const u32* nl, double2* np, double2* nh, hipStream_t sm) {
    typedef Geo<LOGC> G;
    hipLaunchKernelGGL((k_constants_fd<LOGC>), dim3(count), dim3(G::T), G::lds, sm, A, npl, nl, np, nh);
    return hipGetLastError();
}
hipError_t launch_constants(const Args& A, u32 k, u32 count, const u32* npl, const u32* nl, double2* np, double2* nh, hipStream_t sm) {
    switch (k) {
        case 1024: return consts<11>(A, count, npl, nl, np, nh, sm);
        case 2048: return consts<12>(A, count, npl, nl, np, nh, sm);
        case 4096: return consts<13>(A, count, npl, nl, np, nh, sm);
        case 8192: return consts<14>(A, count, npl, nl, np, nh, sm);
        case 16384:
            hipLaunchKernelGGL(k_constants_fd_split, dim3(count), dim3(1024), Geo<14>::lds, sm, A, npl, nl, np, nh, A.dig);
            return hipGetLastError();
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_mul(const Args& A, u32 k, u32 out, u32 a, u32 b, double2* spec, hipStream_t sm) {
    switch (k) {
        case 1024: hipLaunchKernelGGL(k_mul_fd<11>, dim3(1), dim3(Geo<11>::T), Geo<11>::lds, sm, A, out, a, b, spec); break;
        case 2048: hipLaunchKernelGGL(k_mul_fd<12>, dim3(1), dim3(Geo<12>::T), Geo<12>::lds, sm, A, out, a, b, spec); break;
        case 4096: hipLaunchKernelGGL(k_mul_fd<13>, dim3(1), dim3(Geo<13>::T), Geo<13>::lds, sm, A, out, a, b, spec); break;
        case 8192: hipLaunchKernelGGL(k_mul_fd<14>, dim3(1), dim3(Geo<14>::T), Geo<14>::lds, sm, A, out, a, b, spec); break;
        case 16384: hipLaunchKernelGGL(k_mul_fd<15>, dim3(1), dim3(1024), Geo<14>::lds, sm, A, out, a, b, spec); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_plain(const Args& A, u32 k, u32 first, u32 count, u32* out, u32* T, hipStream_t sm) {
    const dim3 g(count);
    switch (k) {
        case 1024: hipLaunchKernelGGL(k_plain_fd<11>, g, dim3(Geo<11>::T), Geo<11>::lds, sm, A, first, out, T); break;
        case 2048: hipLaunchKernelGGL(k_plain_fd<12>, g, dim3(Geo<12>::T), Geo<12>::lds, sm, A, first, out, T); break;
        case 4096: hipLaunchKernelGGL(k_plain_fd<13>, g, dim3(Geo<13>::T), Geo<13>::lds, sm, A, first, out, T); break;
        case 8192: hipLaunchKernelGGL(k_plain_fd<14>, g, dim3(Geo<14>::T), Geo<14>::lds, sm, A, first, out, T); break;
        case 16384: hipLaunchKernelGGL(k_plain_fd<15>, g, dim3(1024), Geo<14>::lds, sm, A, first, out, T); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace fd
}  // namespace mm
