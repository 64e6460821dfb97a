// mm_mx.hip - the matrix-core step kernels of every length they run (L = 16 .. 1,024), in an
// object of their own.

#include "mm_mx.h"

#include <type_traits>

namespace mm {
namespace mx {

template <u32 NB, bool BARE>
__global__ __launch_bounds__(64) void k_steps_mx(Args A, u32 bits) {
    extern __shared__ __align__(16) unsigned char lds[];
    steps<NB, BARE>(A, blockIdx.x, bits, threadIdx.x, lds);
}

template <u32 NB> __global__ __launch_bounds__(64) void k_mul_mx(Args A, u32 out, u32 a, u32 b) {
    extern __shared__ __align__(16) unsigned char lds[];
    product_of<NB>(A, out, a, b, threadIdx.x, lds);
}

template <u32 NB> __global__ __launch_bounds__(64) void k_plain_mx(Args A, u32 first, u32* out) {
    extern __shared__ __align__(16) unsigned char lds[];
    plain<NB>(A, first + blockIdx.x, out + (size_t)blockIdx.x * Slot<NB>::k, threadIdx.x, lds);
}

// k = 8 .. 512 limbs. The limb sums stay below BETA (2^32 - 1) while c n <= 2^20.
bool fits(u32 k, u32 base) { return k >= 8 && k <= 512 && (k & (k - 1)) == 0 && (u64)base * 4 * k <= (1u << 20); }

// Dynamic LDS of a workgroup (one wave): padded so that a whole number of waves per SIMD fits a CU's
// 160 KiB. At L = 1,024 nine waves would fit, one SIMD has three of them and the others wait for it:
// 78 M squarings/s at 4,096 slots against 84 M with eight.
template <u32 NB> static constexpr u32 lds_bytes() {
    constexpr u32 cu = 160 * 1024, per_simd = cu / Lay<NB>::bytes / 4;
    static_assert(per_simd >= 1, "a wave per SIMD");
    return per_simd < 4 ? cu / (4 * per_simd) & ~15u : Lay<NB>::bytes;
}

template <u32 NB> static hipError_t go(const Args& A, u32 slots, u32 bits, bool bare, hipStream_t sm) {
    if (bare)
        hipLaunchKernelGGL((k_steps_mx<NB, true>), dim3(slots), dim3(64), lds_bytes<NB>(), sm, A, bits);
    else
        hipLaunchKernelGGL((k_steps_mx<NB, false>), dim3(slots), dim3(64), lds_bytes<NB>(), sm, A, bits);
    return hipGetLastError();
}

template <class Go> static hipError_t by_length(u32 k, Go&& g) {
    switch (k / 8) {
        case 1: return g(std::integral_constant<u32, 1>());
        case 2: return g(std::integral_constant<u32, 2>());
        case 4: return g(std::integral_constant<u32, 4>());
        case 8: return g(std::integral_constant<u32, 8>());
        case 16: return g(std::integral_constant<u32, 16>());
        case 32: return g(std::integral_constant<u32, 32>());
        case 64: return g(std::integral_constant<u32, 64>());
        default: return hipErrorInvalidValue;
    }
}
hipError_t launch(const Args& A, u32 k, u32 slots, u32 bits, bool bare, hipStream_t sm) {
    return by_length(k, [&](auto nb) { return go<decltype(nb)::value>(A, slots, bits, bare, sm); });
}
hipError_t launch_mul(const Args& A, u32 k, u32 out, u32 a, u32 b, hipStream_t sm) {
    return by_length(k, [&](auto nb) {
        constexpr u32 NB = decltype(nb)::value;
        hipLaunchKernelGGL(k_mul_mx<NB>, dim3(1), dim3(64), Lay<NB>::bytes, sm, A, out, a, b);
        return hipGetLastError();
    });
}
hipError_t launch_plain(const Args& A, u32 k, u32 first, u32 count, u32* out, hipStream_t sm) {
    return by_length(k, [&](auto nb) {
        constexpr u32 NB = decltype(nb)::value;
        hipLaunchKernelGGL(k_plain_mx<NB>, dim3(count), dim3(64), lds_bytes<NB>(), sm, A, first, out);
        return hipGetLastError();
    });
}

}  // namespace mx
}  // namespace mm
