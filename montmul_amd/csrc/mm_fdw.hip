// mm_fdw.hip - the double-precision step at L = 65,536, several workgroups to a slot.
//
// Digits of 16 bits would leave no proof of exactness at this length (C 2^30 127 2^-53 = 0.99), so a
// residue is 131,072 signed digits in base 256: 131,072 2^14 130 2^-53 = 3e-5 (2e-6 found, as in mm_fd.h). As in SplitSlot (mm_fd.h),
// X^C - i is a product of eight X^H - z_p, H = 16,384, z_p = exp(2 pi i (4p + 1) / 32), and the last product,
// right-angled at half the length, of four: z_p = exp(2 pi i (4p + 1) / 16). The parts are independent
// weighted transforms of length H, one workgroup each; the coefficients follow from the parts' results by
// an 8- or 4-point transform across them, H apart.
//
// A step is nine launches, three for each of T = c x^2, m = (T mod R) N' mod R and V = m N mod (R + 1): the
// parts (8, 8 and 4 workgroups of 1,024 threads a slot), the coefficients as limb sums (16 of 256) and the
// carries (one). The launches' ends are what orders the workgroups of a slot: nothing waits inside a kernel.
// Up to 64 slots run together: 512 workgroups of parts fill the chip, and their scratch stays 2.6 MiB
// a slot. What bounds a step is the parts' transforms, one workgroup to a CU for their LDS.
// Measured against the radix-4 kernel (one workgroup a slot, its transforms in HBM) that it replaces by
// default, moduli of 1,000,000 bits, ms a step: 1 slot 1.98 -> 0.17, 16 slots 1.98 -> 0.21, 64 slots
// 2.02 -> 0.43, 256 slots 2.96 -> 1.73. Of the 0.43 the parts take 0.28, the limb sums 0.09 (the parts'
// results are 2 MiB a slot, written and read), the carries 0.06.

#include "mm_fdw.h"

#include <algorithm>

namespace mm {
namespace fdw {

using namespace fd;
constexpr u32 SG = 0x80808080u, T = 1024;
typedef Geo<14> G;
constexpr u32 ROWS_T = 0, ROWS_V = 32, EW_T = 48 * T, EW_V = EW_T + 8 * 16, Z_T = EW_V + 4 * 16, Z_V = Z_T + 8 * 8;

enum { SQUARE, LOW, WRAP, SPEC_LOW, SPEC_WRAP };  // T, m and V; the spectra of N' and N

__device__ __forceinline__ bool done(const Args& A, u32 slot) { return A.pos[slot] >= A.nbits[slot]; }
__device__ __forceinline__ u32 factor(const Args& A, u32 slot) {
    const u32 pos = A.pos[slot];
    return (A.exp[(size_t)slot * A.ew + (pos >> 5)] >> (31 - (pos & 31))) & 1 ? A.base : 1;
}
__device__ __forceinline__ const double2* table(const Args& A, u32 off) {
    u64 w = (u64)(A.tw + off);
    asm volatile("" : "+s"(w));
    return (const double2*)w;
}

// One part of a product: workgroup b does part b % P of slot b / P of the group.
template <int M> __global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4))) void k_parts(Args A) {
    extern __shared__ __align__(16) unsigned char lds[];
    constexpr bool V = M == WRAP || M == SPEC_WRAP;
    constexpr u32 P = V ? 4 : 8;
    const u32 g = blockIdx.x / P, p = blockIdx.x % P, slot = A.first + g;
    if (M <= WRAP && done(A, slot)) return;
    fd::Args fa{};
    fa.w = A.w;
    Slot<14> s(fa, lds);
    {
        const u32* src = M == LOW ? A.lim + (size_t)slot * 3 * K : M == WRAP ? A.lim + (size_t)slot * 3 * K + 2 * K : A.dig + (size_t)g * K;
        const u32 t = tid();
#pragma unroll
        for (u32 i = 0; i < 8; i++) ((uint4*)s.X)[t + T * i] = ((const uint4*)src)[t + T * i];
    }
    __syncthreads();
    Z v[16];
    {
        const u32 t = tid();
        const unsigned char* B = (const unsigned char*)s.X + t;
        const double2 *z = table(A, V ? Z_V + 4 * p : Z_T + 8 * p), *w = table(A, (V ? EW_V : EW_T) + 16 * p);
        auto digit = [&](u32 j) { return (double)(int)(int8_t)(B[j] ^ 0x80); };
#pragma unroll
        for (u32 e = 0; e < 16; e++) {
            Z a{digit(T * e), V ? digit(T * e + 4 * H) : 0.0};
#pragma unroll
            for (u32 q = 1; q < P; q++) {
                const double2 zq = z[q];
                const double d = digit(T * e + q * H);
                a.r = __builtin_fma(d, zq.x, a.r);
                a.i = __builtin_fma(d, zq.y, a.i);
                if constexpr (V) {
                    const double h = digit(T * e + (q + 4) * H);
                    a.r = __builtin_fma(h, -zq.y, a.r);
                    a.i = __builtin_fma(h, zq.x, a.i);
                }
            }
            if (M == SQUARE && e == 0 && t == 0) a.i += (double)A.fl[2 * g];  // digit C, where X^C = i
            const double2 we = w[e];
            v[e] = mulw<false>(a, we.x, we.y);
            fence();
        }
    }
    settle(v);
    __syncthreads();
    const double2* rows = A.tw + T * ((V ? ROWS_V : ROWS_T) + 4 * p);
    forward<14, 14>(v, A.w, lds, true, rows);
    if constexpr (M == SPEC_LOW || M == SPEC_WRAP) {
        double2* o = (V ? A.n : A.np) + ((size_t)slot * P + p) * H + tid();
#pragma unroll
        for (u32 e = 0; e < 16; e++) o[T * e] = make_double2(v[e].r, v[e].i);
        return;
    }
    if constexpr (M == SQUARE) {
#pragma unroll
        for (u32 e = 0; e < 16; e++) v[e] = Z{(v[e].r + v[e].i) * (v[e].r - v[e].i), 2.0 * v[e].r * v[e].i};
    } else
        Spectrum<T>((V ? A.n : A.np) + ((size_t)slot * P + p) * H, tid()).apply(v);
    settle(v);
    inverse<14, 14>(v, A.w, lds, true, rows);
    const double2* w = table(A, (V ? EW_V : EW_T) + 16 * p);
    double2* o = A.part + ((size_t)g * 8 + p) * H + tid();
#pragma unroll
    for (u32 e = 0; e < 16; e++) {
        const double2 we = w[e];
        const Z z = mulw<true>(v[e], we.x, we.y);
        o[T * e] = make_double2(z.r, z.i);
        if (e % 4 == 3) fence();
    }
}

// The limb sums of a product from its parts: thread j of the 4,096 of a slot takes the parts' elements
// 4j .. 4j + 3, a limb of each block of H digits.
template <int M> __global__ __launch_bounds__(256) void k_sums(Args A) {
    constexpr u32 P = M == WRAP ? 4 : 8;
    const u32 g = blockIdx.x / 16, j = blockIdx.x % 16 * 256 + threadIdx.x;
    if (done(A, A.first + g)) return;
    const double2* in = A.part + (size_t)g * 8 * H + 4 * j;
    Z a[4][P];
#pragma unroll
    for (u32 p = 0; p < P; p++)
#pragma unroll
        for (u32 d = 0; d < 4; d++) {
            const double2 v = in[p * H + d];
            a[d][p] = Z{v.x, v.y};
        }
    const double2* z = table(A, M == WRAP ? Z_V : Z_T);  // part 0's: z_0^q
    u64 re[P] = {}, im[P] = {};
#pragma unroll
    for (u32 d = 0; d < 4; d++) {
        Z* v = a[d];
        if constexpr (P == 4)
            dft4<true>(v[0], v[1], v[2], v[3]);
        else {
            dft4<true>(v[0], v[2], v[4], v[6]);
            dft4<true>(v[1], v[3], v[5], v[7]);
            const Z e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
            const Z o0 = v[1], o1 = mul_w2<true>(v[3]), o2 = rot<true>(v[5]), o3 = rot<true>(mul_w2<true>(v[7]));
            v[0] = e0 + o0; v[4] = e0 - o0;
            v[1] = e1 + o1; v[5] = e1 - o1;
            v[2] = e2 + o2; v[6] = e2 - o2;
            v[3] = e3 + o3; v[7] = e3 - o3;
        }
        auto whole = [](double f) { return __builtin_bit_cast(u64, __builtin_fma(f, 1.0 / (P * H), MAGIC)) - MAGIC_BITS; };
#pragma unroll
        for (u32 q = 0; q < P; q++) {
            Z c = v[q];
            if (q) {
                const double2 zq = z[q];
                c = mulw<true>(c, zq.x, zq.y);
            }
            re[q] += whole(c.r) << (8 * d);
            if (M != LOW) im[q] += whole(c.i) << (8 * d);
        }
    }
    i64* o = A.sum + (size_t)g * 2 * K + j;
#pragma unroll
    for (u32 q = 0; q < P; q++) {
        o[q * (H / 4)] = (i64)re[q];
        if (M != LOW) o[(P + q) * (H / 4)] = (i64)im[q];
    }
}

// 8,192 sums through the carry into biased limbs at dst, `in` at the lowest; returns the carry out.
__device__ __forceinline__ u32 carry_chunk(const i64* sum, u32 c, u32 in, u32* dst, u32* sc) {
    const u32 t = tid();
    u64 s[8];
    u32 l[8];
#pragma unroll
    for (u32 i = 0; i < 8; i++) s[i] = (u64)(sum[8 * t + i] * (i64)c) + BIAS + SG;
    if (t == 0) s[0] += in;
    const u32 out = bcarry<16>(s, l, sc, t);
    ((uint4*)(dst + 8 * t))[0] = make_uint4(l[0], l[1], l[2], l[3]);
    ((uint4*)(dst + 8 * t))[1] = make_uint4(l[4], l[5], l[6], l[7]);
    __syncthreads();
    return out;
}
// The carries of a product, one workgroup a slot; WRAP ends the step (see Slot::step).
template <int M> __global__ __launch_bounds__(1024) void k_carry(Args A) {
    extern __shared__ __align__(16) u32 words[];  // WRAP: x's biased limbs
    __shared__ u32 sc[32], flag[2];
    const u32 g = blockIdx.x, slot = A.first + g;
    if (done(A, slot)) return;
    const i64* sum = A.sum + (size_t)g * 2 * K;
    u32 *Tl = A.lim + (size_t)slot * 3 * K, *md = Tl + 2 * K, *fl = A.fl + 2 * g;
    u32 bad = 0;
    if constexpr (M == SQUARE) {
        const u32 c = factor(A, slot), up = c * fl[0];  // fl[0]^2 = fl[0]
        u32 in = (u32)BETA + up;
        for (u32 q = 0; q < 2 * K; q += 8192) in = carry_chunk(sum + q, c, in, Tl + q, sc);
        u32 et = in - (u32)BETA + up;
        if (et != 0) {  // T = T' + et R^2: only T' < 0 with et = 1 stands for a number below R^2
            if (tid() < 64) flag[1] = sign_of<SG>(Tl, 2 * K) & 1;
            __syncthreads();
            bad = et != flag[1];
            et = flag[1];
        }
        if (tid() == 0) fl[1] = et;
    } else if constexpr (M == LOW) {
        u32 in = (u32)BETA;
        for (u32 q = 0; q < K; q += 8192) in = carry_chunk(sum + q, 1, in, md + q, sc);
        if (tid() < 64 && sign_of<SG>(md, K) == 1 && tid() == 0) add_small(md, K, -1);  // m = m' + R = m' - 1
    } else {
        const u32 et = fl[1];
        u32 in = (u32)BETA - et;
        for (u32 q = 0; q < K; q += 8192) {
            const u32 t = tid();
            const u32* p = Tl + q + 8 * t;
            u64 s[8];
            u32 l[8];
#pragma unroll
            for (u32 i = 0; i < 8; i++) s[i] = (u64)((i64)p[K + i] - (i64)p[i] - sum[q + 8 * t + i]) + BIAS + SG;
            if (t == 0) s[0] += in;
            in = bcarry<16>(s, l, sc, t);
            uint4* w = (uint4*)(words + q + 8 * t);
            w[0] = make_uint4(l[0], l[1], l[2], l[3]);
            w[1] = make_uint4(l[4], l[5], l[6], l[7]);
            __syncthreads();
        }
        u32 ex = 0;
        bad = fix_number<SG, T>(words, K, in - (u32)BETA, et, Tl, flag, ex);
        __syncthreads();
        uint4* o = (uint4*)(A.dig + (size_t)g * K);
        const u32 t = tid();
#pragma unroll
        for (u32 i = 0; i < 8; i++) o[t + T * i] = ((const uint4*)words)[t + T * i];
        if (t == 0) {
            fl[0] = ex;
            A.pos[slot]++;
        }
    }
    if (bad) A.err[slot] = 1;
}

// K limbs of each slot of the group at src as biased digits, with the flag of what stands above them;
// wrapped: modulo R + 1 instead.
__global__ __launch_bounds__(1024) void k_digits(Args A, const u32* src, u32 wrapped) {
    __shared__ u32 sc[32];
    const u32 g = blockIdx.x;
    u32* dig = A.dig + (size_t)g * K;
    u32 in = 0;
    for (u32 q = 0; q < K; q += 8192) {
        const u32 t = tid();
        const u32* p = src + (size_t)g * K + q + 8 * t;
        u64 s[8];
        u32 l[8];
#pragma unroll
        for (u32 i = 0; i < 8; i++) s[i] = (u64)p[i] + SG;
        if (t == 0) s[0] += in;
        in = bcarry<16>(s, l, sc, t);
#pragma unroll
        for (u32 i = 0; i < 8; i++) dig[q + 8 * t + i] = l[i];
        __syncthreads();
    }
    if (tid() == 0) {
        A.fl[2 * g] = in;
        if (wrapped && in) add_small(dig, K, -1);
    }
}
// x's limbs from its digits.
__global__ __launch_bounds__(1024) void k_limbs(Args A) {
    __shared__ u32 sc[32];
    const u32 g = blockIdx.x;
    const u32* dig = A.dig + (size_t)g * K;
    u32* x = A.x + (size_t)(A.first + g) * K;
    u32 in = 1;
    for (u32 q = 0; q < K; q += 8192) {
        const u32 t = tid();
        u64 s[8];
        u32 l[8];
#pragma unroll
        for (u32 i = 0; i < 8; i++) s[i] = (u64)dig[q + 8 * t + i] + (0xffffffffu - SG);
        if (t == 0) s[0] += in;
        in = bcarry<16>(s, l, sc, t);
#pragma unroll
        for (u32 i = 0; i < 8; i++) x[q + 8 * t + i] = l[i];
        __syncthreads();
    }
}

// Limb sums stay below BETA (2^32 - 1): c (2^31 + 2^8) (2^24 + 2^16 + 2^8 + 1) with c < 128.
static_assert((unsigned __int128)127 * ((1ull << 31) + 256) * 0x1010101u < BIAS, "c < 128");
bool fits(u32 k, u32 base) { return k == K && base < 128; }

void make_tables(double2* out) {
    fd::make_tables(H, out);
    out += fd::table_elems(H);
    for (u64 p = 0; p < 8; p++)
        for (u64 a = 0; a < 4; a++)
            for (u64 t = 0; t < T; t++) out[(ROWS_T + 4 * p + a) * T + t] = unit(t * (128 * a + 4 * p + 1), 32ull * H);
    for (u64 p = 0; p < 4; p++)
        for (u64 a = 0; a < 4; a++)
            for (u64 t = 0; t < T; t++) out[(ROWS_V + 4 * p + a) * T + t] = unit(t * (64 * a + 4 * p + 1), 16ull * H);
    for (u64 p = 0; p < 8; p++)
        for (u64 e = 0; e < 16; e++) out[EW_T + 16 * p + e] = unit((4 * p + 1) * e, 512);
    for (u64 p = 0; p < 4; p++)
        for (u64 e = 0; e < 16; e++) out[EW_V + 16 * p + e] = unit((4 * p + 1) * e, 256);
    for (u64 p = 0; p < 8; p++)
        for (u64 q = 0; q < 8; q++) out[Z_T + 8 * p + q] = unit((4 * p + 1) * q, 32);
    for (u64 p = 0; p < 4; p++)
        for (u64 q = 0; q < 4; q++) out[Z_V + 4 * p + q] = unit((4 * p + 1) * q, 16);
}

hipError_t set_lds_limit() {
    for (const void* k : {(const void*)k_parts<SQUARE>, (const void*)k_parts<LOW>, (const void*)k_parts<WRAP>, (const void*)k_parts<SPEC_LOW>,
                          (const void*)k_parts<SPEC_WRAP>}) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)G::lds);
        if (e != hipSuccess) return e;
    }
    return hipFuncSetAttribute((const void*)k_carry<WRAP>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(4 * K));
}

template <int M> static void product(const Args& A, u32 slots, hipStream_t sm) {
    hipLaunchKernelGGL(k_parts<M>, dim3(slots * (M == WRAP ? 4 : 8)), dim3(T), G::lds, sm, A);
    hipLaunchKernelGGL(k_sums<M>, dim3(slots * 16), dim3(256), 0, sm, A);
    hipLaunchKernelGGL(k_carry<M>, dim3(slots), dim3(T), M == WRAP ? 4 * K : 0, sm, A);
}
hipError_t launch(Args A, u32 slots, const u32* steps, hipStream_t sm) {
    for (A.first = 0; A.first < slots; A.first += GROUP) {
        const u32 c = std::min(GROUP, slots - A.first), bits = steps[A.first / GROUP];
        if (bits == 0) continue;
        hipLaunchKernelGGL(k_digits, dim3(c), dim3(T), 0, sm, A, A.x + (size_t)A.first * K, 0u);
        for (u32 i = 0; i < bits; i++) {
            product<SQUARE>(A, c, sm);
            product<LOW>(A, c, sm);
            product<WRAP>(A, c, sm);
            if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(k_limbs, dim3(c), dim3(T), 0, sm, A);
    }
    return hipGetLastError();
}
hipError_t launch_constants(Args A, u32 count, const u32* npl, const u32* nl, hipStream_t sm) {
    for (u32 i = 0; i < count; i += GROUP, A.first += GROUP) {
        const u32 c = std::min(GROUP, count - i);
        hipLaunchKernelGGL(k_digits, dim3(c), dim3(T), 0, sm, A, npl + (size_t)i * K, 0u);
        hipLaunchKernelGGL(k_parts<SPEC_LOW>, dim3(8 * c), dim3(T), G::lds, sm, A);
        hipLaunchKernelGGL(k_digits, dim3(c), dim3(T), 0, sm, A, nl + (size_t)i * K, 1u);
        hipLaunchKernelGGL(k_parts<SPEC_WRAP>, dim3(4 * c), dim3(T), G::lds, sm, A);
    }
    return hipGetLastError();
}

}  // namespace fdw
}  // namespace mm
