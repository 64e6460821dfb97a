// mm_fd.h - the Montgomery step on double-precision transforms (wraparound path, L = 2,048 ..
// 32,768, k = L / 2 limbs).
//
// A residue is C = L signed digits of 16 bits (-2^15 .. 2^15), in double precision, which issues one
// multiply-add a cycle per lane where a product in GF(M61^2) takes sixteen 64-bit multiply-adds
// and their folds. Products are weighted ("right-angle") transforms: a_j + i a_(j+C) times
// zeta^j, zeta = exp(i pi / 2C), cyclic length C, gives products modulo X^2C + 1. Coefficients are
// integers and are rounded to the nearest one.
//
// Exactness. With u = 2^-53, along each path from an input to an output of a transform a radix-16 pass
// adds a relative error of at most 4 u (four levels of sums) and 2 x 3 u (its inner rotations), each of
// the four twiddle factors between passes and the weights 3.3 u (tables within u / 2), the last
// radix-2 or 4 stage 2 u: e = 49 u a transform. What that makes of a coefficient of a b, with A and B the
// spectra, of length n and of 2-norms sqrt(n) |a| and sqrt(n) |b|:
//   - the forward transforms' errors, at most e sqrt(n) |a| in the 2-norm (every pass is a multiple of a unitary
//     one), reach a coefficient as 1/n sum |dA_j| |B_j| <= e |a| |b| each (Cauchy and Schwarz);
//   - the inverse's error at an output is at most e times the sum of what its paths bring there,
//     1/n sum |A_j B_j| <= |a| |b|, and so is the pointwise product's, with 3 u. (A bound by the 2-norm of a b would
//     not do: that can be sqrt(C) |a| |b|.)
// In all 150 u |a| |b| <= C 2^30 150 2^-53: 0.04, 0.07, 0.15 and 0.29 at L = 2,048, 4,096,
// 8,192 and 16,384, below the 0.5 that rounding needs, for any digits (SplitSlot counts L = 32,768). The
// farthest from an integer that a copy of these kernels that keeps the largest distance found:
// L = 2,048 / 4,096 / 8,192 / 16,384 / 32,768: 5e-5 / 6e-5 / 9e-5 / 1.2e-4 / 2.4e-4 on random moduli, 0.0012 / 0.0024 /
// 0.006 / 0.012 / 0.023 on digits of the largest size with equal, alternating and other periodic signs.
//
// A step, R = 2^(32k) = 2^(16 C):
//     T = c x^2                  transform of length C, square, inverse
//     m = (T mod R) N' mod R     transform, product with N''s spectrum, inverse (low half)
//     V = m N mod (R + 1)        negacyclic: weighted transforms of length C / 2
//     x = (T + m N) / R          = floor(T / R) - (T mod R) - V mod (R + 1), since R = -1 there
// so the last product needs half the length and no low half. Signed digits are number + 0x8000 in
// every digit, carried as an ordinary number, then each digit xor 0x8000 (see mm_mx.h).
//
// One workgroup of C / 16 threads steps one slot, 16 elements per thread in registers. Passes of
// radix 16 have strides C/16, C/256 and C/4096; the last factor of 1, 2 or 4 is taken across
// neighbouring lanes. Only the exchange after the first pass crosses waves; all go through LDS one
// component at a time (8 bytes per element), so that two workgroups share a CU at L = 8,192 beside
// the later passes' twiddles, which stay in LDS.
//
// Measured against the modular transforms (mm_v2.h) that it replaces by default: L = 2,048 (2,048
// slots) 14.4 -> 36 M squarings/s (30 M on the matrix cores, whose work grows as n^2; at 1,024 they
// do 91 M, and this step, by its work, 75 M), 4,096 (1,024 slots) 7.0 -> 15.7 M, 8,192 (4,096
// slots) 3.6 -> 9.1 M, 16,384 (1,024 slots) 1.31 -> 3.7 M, 32,768 (1,024 slots) 0.42 -> 1.18 M;
// one slot alone at 8,192 92 -> 34 us a step, at 32,768 560 -> 147 us.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mm {
namespace fd {

typedef uint32_t u32;
typedef uint64_t u64;
typedef int64_t i64;
typedef uint16_t u16;

constexpr u32 SGN = 0x80008000u;
constexpr u64 BETA = 0x7fffffffu;  // |limb sums| < BETA (2^32 - 1): c C < 2^17 (fits)
constexpr u64 BIAS = BETA * 0xffffffffull;
// A limb's sum is c (v + 2^16 w), v and w coefficients: of C + 1 digits, the highest 0 or 1, so at most
// C 2^30 + 2^16. Biased (and with T's limbs, for x) it stays below 2^64 with a carry from below.
constexpr bool sums_fit(u64 c, u64 C) {
    const unsigned __int128 most = (unsigned __int128)c * ((C << 30) + 65536) * 65537;
    return most < BIAS && most + BIAS + SGN + BETA + 0xffffffffull < (unsigned __int128)1 << 64;
}
static_assert(sums_fit(131071 / 2048, 2048) && sums_fit(131071 / 4096, 4096) && sums_fit(131071 / 8192, 8192) &&
                  sums_fit(131071 / 16384, 16384) && sums_fit(131071 / 32768, 32768),
              "c C < 2^17");
constexpr double MAGIC = 6755399441055744.0;  // 1.5 2^52: integers appear in the low bits of the sum
constexpr u64 MAGIC_BITS = 0x4338000000000000ull;

// Twiddles of one complex length C (host: make_tables), T = C / 16. The transforms of length C / 2
// use every other element of them.
struct Tables {
    const double2* t0;  // pass 0 and the weights: exp(2 pi i t (16 a + 1) / 4C) at a T + t, a < 4, then
                        // exp(2 pi i t b / C) at (3 + b) T + t, b = 1 .. 3: element 4 a + b takes both
    const double2* t1;  // pass 1: exp(2 pi i j m / (C/16)) at m C/256 + j
    const double2* t2;  // pass 2: exp(2 pi i j m / (C/256)) at m C/4096 + j
    // The split length 2C (see SplitSlot): t0's first four rows with the parts' weights, four rows for
    // each part p, exp(2 pi i t (32 a + 4 p + 1) / 8C), then exp(2 pi i (4 p + 1) e / 128) at 16 p + e.
    const double2* ts;
};

struct Args {
    Tables w;           // length C = 2k (k = 16,384: C = k, the parts' length)
    u32* x;             // k limbs per slot
    const double2* np;  // 2k per slot: spectrum of N', at e C/16 + t (k = 16,384: part after part)
    const double2* n;   // k per slot: spectrum of N (length k)
    double2* part;      // k = 16,384: k per slot, the first part's result
    u32* dig;           // k = 16,384: k per slot, the digits that the second part loads again
    const u32* exp;     // ew words per slot, most significant bit first
    const u32* nbits;
    u32* pos;
    u32* err;
    u32* lim;           // T (2k limbs) at 3k limbs per slot; run_bare leaves it as a number
    u32 ew, base;
};

template <u32 LOGC> struct Geo {
    static constexpr u32 C = 1u << LOGC, T = C / 16, k = C / 2, waves = T / 64;
    static constexpr u32 S1 = C / 256;                          // pass 1's stride
    static constexpr u32 R = C >= 4096 ? C / 4096 : 1;          // pass 2's stride, the factor across lanes
    static constexpr u32 R2 = C / 4096;                         // columns of pass 2's twiddles
    // LDS: the exchange buffer (doubles), passes 1 and 2's twiddles, carry scratch, flags.
    static constexpr u32 xwords = C + C / 16;
    static constexpr u32 o1 = xwords * 8, o2 = o1 + 256 * S1, osc = o2 + 256 * R2, lds = osc + 3 * 32 * 4 + 16;
    static_assert(LOGC >= 10 && LOGC <= 14, "1,024 <= C <= 16,384");
    // Exchange position: 16 R elements and R of padding, which spreads the strides of the second
    // exchange over the banks.
    static __device__ __forceinline__ u32 at(u32 p) { return p + R * (p / (16 * R)); }
};
// The thread's index, read anew at each phase: an index kept from phase to phase would keep every
// phase's address arithmetic in registers across the whole step.
__device__ __forceinline__ u32 tid() {
    u32 t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}
// Keeps the scheduler from moving later phases' loads up, whose registers the step does not have.
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

__device__ __forceinline__ void wsync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

struct Z { double r, i; };
// Ends a phase: the elements are computed here, and not sunk past the barriers, waits and loads that
// follow.
__device__ __forceinline__ void settle(Z* v) {
#pragma unroll
    for (int e = 0; e < 16; e++) asm volatile("" : "+v"(v[e].r), "+v"(v[e].i));
    fence();
}
__device__ __forceinline__ Z operator+(Z a, Z b) { return Z{a.r + b.r, a.i + b.i}; }
__device__ __forceinline__ Z operator-(Z a, Z b) { return Z{a.r - b.r, a.i - b.i}; }
// a w, or a conj(w).
template <bool INV> __device__ __forceinline__ Z mulw(Z a, double wr, double wi) {
    if (INV) wi = -wi;
    return Z{__builtin_fma(a.r, wr, -(a.i * wi)), __builtin_fma(a.r, wi, a.i * wr)};
}
template <bool INV> __device__ __forceinline__ Z rot(Z a) { return INV ? Z{a.i, -a.r} : Z{-a.i, a.r}; }  // by +-i
constexpr double C1 = 0.92387953251128675613, S1 = 0.38268343236508977173, RH = 0.70710678118654752440;

// 4-point transform, in place, natural order.
template <bool INV> __device__ __forceinline__ void dft4(Z& a, Z& b, Z& c, Z& d) {
    const Z s0 = a + c, d0 = a - c, s1 = b + d, d1 = rot<INV>(b - d);
    a = s0 + s1;
    c = s0 - s1;
    b = d0 + d1;
    d = d0 - d1;
}
template <bool INV> __device__ __forceinline__ Z mul_w2(Z a) {  // by exp(+-i pi / 4)
    return INV ? Z{(a.r + a.i) * RH, (a.i - a.r) * RH} : Z{(a.r - a.i) * RH, (a.r + a.i) * RH};
}
// 16-point transform in place: v[e] -> sum_e v[e] w^(e m) at v[m].
template <bool INV> __device__ __forceinline__ void dft16(Z* v) {
    // e = e1 + 4 e2, m = 4 m1 + m2: over e2 first, then the twiddles w^(e1 m2), then over e1.
#pragma unroll
    for (u32 e1 = 0; e1 < 4; e1++) dft4<INV>(v[e1], v[e1 + 4], v[e1 + 8], v[e1 + 12]);  // m2 at v[e1 + 4 m2]
    v[1 + 4] = mulw<INV>(v[1 + 4], C1, S1);
    v[2 + 4] = mul_w2<INV>(v[2 + 4]);
    v[3 + 4] = mulw<INV>(v[3 + 4], S1, C1);
    v[1 + 8] = mul_w2<INV>(v[1 + 8]);
    v[2 + 8] = rot<INV>(v[2 + 8]);
    v[3 + 8] = rot<INV>(mul_w2<INV>(v[3 + 8]));
    v[1 + 12] = mulw<INV>(v[1 + 12], S1, C1);
    v[2 + 12] = rot<INV>(mul_w2<INV>(v[2 + 12]));
    v[3 + 12] = mulw<INV>(v[3 + 12], -C1, -S1);
#pragma unroll
    for (u32 m2 = 0; m2 < 4; m2++) dft4<INV>(v[4 * m2], v[4 * m2 + 1], v[4 * m2 + 2], v[4 * m2 + 3]);  // m1 at v[4 m2 + m1]
    // v[4 m2 + m1] holds m = 4 m1 + m2: transpose by renaming.
#pragma unroll
    for (u32 a = 0; a < 4; a++)
#pragma unroll
        for (u32 b = a + 1; b < 4; b++) {
            const Z t = v[4 * a + b];
            v[4 * a + b] = v[4 * b + a];
            v[4 * b + a] = t;
        }
}

// 8-point transform in place: v[e] -> sum_e v[e] w^(e m), at some fixed order of m; the inverse takes
// that order back (both leave the same spectrum position to the same register).
template <bool INV> __device__ __forceinline__ void dft8(Z* v) {
    if constexpr (!INV) {
#pragma unroll
        for (u32 e = 0; e < 4; e++) {
            const Z a = v[e], b = v[e + 4];
            v[e] = a + b;
            v[e + 4] = a - b;
        }
        v[5] = mul_w2<false>(v[5]);
        v[6] = rot<false>(v[6]);
        v[7] = rot<false>(mul_w2<false>(v[7]));
        dft4<false>(v[0], v[1], v[2], v[3]);
        dft4<false>(v[4], v[5], v[6], v[7]);
    } else {
        dft4<true>(v[0], v[1], v[2], v[3]);
        dft4<true>(v[4], v[5], v[6], v[7]);
        v[5] = mul_w2<true>(v[5]);
        v[6] = rot<true>(v[6]);
        v[7] = rot<true>(mul_w2<true>(v[7]));
#pragma unroll
        for (u32 e = 0; e < 4; e++) {
            const Z a = v[e], b = v[e + 4];
            v[e] = a + b;
            v[e + 4] = a - b;
        }
    }
}

// exp(i pi e / 32): the weights of a thread's elements relative to its first.
__device__ constexpr double WC[16] = {1.0, 0.99518472667219688624, 0.98078528040323044913, 0.95694033573220886494,
    0.92387953251128675613, 0.88192126434835502971, 0.83146961230254523708, 0.77301045336273696081,
    0.70710678118654752440, 0.63439328416364549822, 0.55557023301960222474, 0.47139673682599764856,
    0.38268343236508977173, 0.29028467725446236764, 0.19509032201612826785, 0.09801714032956060199};
__device__ __forceinline__ constexpr double wre(u32 e) { return WC[e]; }
__device__ __forceinline__ constexpr double wim(u32 e) { return e == 0 ? 0.0 : WC[16 - e]; }

template <u32 CTRL> __device__ __forceinline__ double dpp(double v) {
    const u64 b = __builtin_bit_cast(u64, v);
    const u32 lo = (u32)__builtin_amdgcn_update_dpp(0, (int)(u32)b, CTRL, 0xf, 0xf, true);
    const u32 hi = (u32)__builtin_amdgcn_update_dpp(0, (int)(u32)(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, (u64)hi << 32 | lo);
}
// The last factor R, across R neighbouring lanes (element j of a group in lane j).
template <u32 R, bool INV> __device__ __forceinline__ void across(Z* v, u32 t) {
    if constexpr (R == 1) return;
    const double s1 = t & 1 ? -1.0 : 1.0;
    if constexpr (R == 2) {
#pragma unroll
        for (u32 e = 0; e < 16; e++)
            v[e] = Z{__builtin_fma(s1, v[e].r, dpp<0xB1>(v[e].r)), __builtin_fma(s1, v[e].i, dpp<0xB1>(v[e].i))};
    }
    if constexpr (R == 4) {
        const double s2 = t & 2 ? -1.0 : 1.0;
        // Selected by component: a choice between two Z went through scratch memory (1.84 M squarings/s
        // at L = 16,384 and 256 slots against 3.5 M).
        const bool l3 = (t & 3) == 3;
#pragma unroll
        for (u32 e = 0; e < 16; e++) {
            Z a = v[e];
            if constexpr (!INV) {
                a = Z{__builtin_fma(s2, a.r, dpp<0x4E>(a.r)), __builtin_fma(s2, a.i, dpp<0x4E>(a.i))};
                const Z b = rot<false>(a);
                a = Z{l3 ? b.r : a.r, l3 ? b.i : a.i};
                a = Z{__builtin_fma(s1, a.r, dpp<0xB1>(a.r)), __builtin_fma(s1, a.i, dpp<0xB1>(a.i))};
            } else {
                a = Z{__builtin_fma(s1, a.r, dpp<0xB1>(a.r)), __builtin_fma(s1, a.i, dpp<0xB1>(a.i))};
                const Z b = rot<true>(a);
                a = Z{l3 ? b.r : a.r, l3 ? b.i : a.i};
                a = Z{__builtin_fma(s2, a.r, dpp<0x4E>(a.r)), __builtin_fma(s2, a.i, dpp<0x4E>(a.i))};
            }
            v[e] = a;
        }
    }
}

typedef double d2 __attribute__((ext_vector_type(2)));

// An element of global memory at a workgroup-uniform address plus the lane's byte offset.
__device__ __forceinline__ d2 ldg(u64 base, u32 off) {
    typedef const __attribute__((address_space(1))) d2* Global;
    return *(Global)(base + off);
}

// Pass 0's twiddles and the weights, as products of two table elements: seven loads, issued ahead
// of the butterfly, where sixteen have to be waited for in four groups.
template <bool INV, u32 T, u32 SUB> struct Twiddle0 {
    d2 w[7];
    // t0: all rows; weighted: the first four, another length's weights in them or not.
    __device__ __forceinline__ Twiddle0(const double2* t0, const double2* weighted, u32 t) {
        u64 a = (u64)weighted, b = (u64)t0;
        asm volatile("" : "+s"(a), "+s"(b));  // or each step's row addresses stay in scalar registers
#pragma unroll
        for (u32 r = 0; r < 7; r++) w[r] = ldg((r < 4 ? a : b) + 16 * SUB * T * r, 16 * SUB * t);
        fence();
    }
    __device__ __forceinline__ void apply(Z* v) const {
#pragma unroll
        for (u32 m = 0; m < 16; m++) {
            if (m % 4) v[m] = mulw<INV>(v[m], w[3 + m % 4].x, w[3 + m % 4].y);
            v[m] = mulw<INV>(v[m], w[m / 4].x, w[m / 4].y);
        }
        fence();
    }
};
// The later passes' twiddles, from LDS: v[m] by tab[m stride], m >= 1.
template <bool INV> __device__ __forceinline__ void twiddle(Z* v, const d2* tab, u32 stride) {
#pragma unroll
    for (u32 g = 0; g < 16; g += 4) {
        d2 w[4];
#pragma unroll
        for (u32 m = 0; m < 4; m++)
            if (g + m) w[m] = tab[(g + m) * stride];
#pragma unroll
        for (u32 m = 0; m < 4; m++)
            if (g + m) v[g + m] = mulw<INV>(v[g + m], w[m].x, w[m].y);
        if (g % 8) fence();
    }
}
// v[e] times a slot's spectrum (HBM), rows of T: eight loads in flight.
template <u32 T> struct Spectrum {
    u64 base;
    u32 off;
    d2 w[8];
    __device__ __forceinline__ Spectrum(const double2* p, u32 t) : base((u64)p), off(16 * t) {
        asm volatile("" : "+s"(base));
#pragma unroll
        for (u32 e = 0; e < 8; e++) w[e] = ldg(base + 16 * T * e, off);
        fence();
    }
    __device__ __forceinline__ void apply(Z* v) {
#pragma unroll
        for (u32 e = 0; e < 8; e++) {
            v[e] = mulw<false>(v[e], w[e].x, w[e].y);
            w[e] = ldg(base + 16 * T * (e + 8), off);
            fence();
        }
#pragma unroll
        for (u32 e = 0; e < 8; e++) v[e + 8] = mulw<false>(v[e + 8], w[e].x, w[e].y);
        fence();
    }
};

// Buffer positions of a thread's elements S apart, relative to the first: with the padding (16 R
// divides S, or S divides 16, R = 1 and the first is below S in its block), or within one block.
constexpr u32 WITHIN = 1u << 31;
__device__ __forceinline__ constexpr u32 spaced(u32 S, u32 e) { return S & WITHIN ? (S & ~WITHIN) * e : S * e + S * e / 16; }
// Exchange of one component at a time: element e written at w + spaced(WS, e), read at
// r + spaced(RS, e). BLOCK: across waves (barriers), else within the wave's own part of the buffer.
template <bool BLOCK, u32 WS, u32 RS> __device__ __forceinline__ void exchange(Z* v, double* X, u32 w, u32 r, bool on) {
    auto sync = [] {
        fence();
        if (BLOCK) __syncthreads();
        else wsync();
        fence();
    };
    fence();
    if (on)
#pragma unroll
        for (u32 e = 0; e < 16; e++) X[w + spaced(WS, e)] = v[e].r;
    sync();
    if (on)
#pragma unroll
        for (u32 e = 0; e < 16; e++) v[e].r = X[r + spaced(RS, e)];
    sync();
    if (on)
#pragma unroll
        for (u32 e = 0; e < 16; e++) X[w + spaced(WS, e)] = v[e].i;
    sync();
    if (on)
#pragma unroll
        for (u32 e = 0; e < 16; e++) v[e].i = X[r + spaced(RS, e)];
    fence();
}

// Positions of thread t's elements: pass 0 at t + T e, pass 1 at p1 + S1 e, pass 2 at p2 + R e. At
// C = 2,048 and 1,024 pass 2 is two 8-point or four 4-point transforms of neighbours. x0, x1, x2: the
// first one's position in the buffer.
template <u32 LOGC> struct Pos {
    typedef Geo<LOGC> G;
    static constexpr u32 X0 = G::T, X1 = G::S1, X2 = G::R | WITHIN;  // spacings of the passes' elements
    u32 t, j1, j2, x0, x1, x2;
    __device__ __forceinline__ explicit Pos(u32 t_) : t(t_) {
        constexpr u32 R = G::R, S1 = G::S1;
        const u32 b = t / S1, i = t % S1;
        j1 = i;
        j2 = i % R;
        x0 = G::at(t);
        x1 = G::at(16 * S1 * b + i);
        x2 = G::at(16 * S1 * b + 16 * R * (i / R) + j2);
    }
};

// Pass 2's butterflies: one of 16 points, or two of 8 or four of 4 where no more are left.
template <u32 LOGC, bool INV> __device__ __forceinline__ void last16(Z* v) {
    if constexpr (LOGC >= 12)
        dft16<INV>(v);
    else if constexpr (LOGC == 10) {
#pragma unroll
        for (u32 g = 0; g < 16; g += 4) dft4<INV>(v[g], v[g + 1], v[g + 2], v[g + 3]);
    } else {
        dft8<INV>(v);
        dft8<INV>(v + 8);
    }
}

// Forward transform of weighted elements in pass-0 layout (the thread's own weights exp(i pi e / 32)
// already applied); the spectrum ends in pass-2 layout. LOGF: the tables' length. The buffer must be
// free (barrier before).
template <u32 LOGF, u32 LOGC>
__device__ __forceinline__ void forward(Z* v, const Tables& W, unsigned char* lds, bool on, const double2* weighted) {
    typedef Geo<LOGC> G;
    typedef Geo<LOGF> F;
    typedef Pos<LOGC> P;
    constexpr u32 SUB = 1u << (LOGF - LOGC);
    double* X = (double*)lds;
    if (on) {
        const Twiddle0<false, G::T, SUB> f(W.t0, weighted, tid());
        dft16<false>(v);
        settle(v);
        f.apply(v);
        settle(v);
    }
    {
        const P p(tid());
        exchange<true, P::X0, P::X1>(v, X, p.x0, p.x1, on);
    }
    if (on) {
        dft16<false>(v);
        settle(v);
        twiddle<false>(v, (const d2*)(lds + F::o1) + SUB * P(tid()).j1, F::S1);
        settle(v);
        {
            const P p(tid());
            exchange<false, P::X1, P::X2>(v, X, p.x1, p.x2, true);
        }
        last16<LOGC, false>(v);
        settle(v);
        if constexpr (G::R > 1) {
            twiddle<false>(v, (const d2*)(lds + F::o2) + SUB * P(tid()).j2, F::R2);
            settle(v);
            across<G::R, false>(v, tid());
            settle(v);
        }
    }
}
// Its inverse up to the thread's own weights and the factor C: pass-2 layout in, pass-0 out.
template <u32 LOGF, u32 LOGC>
__device__ __forceinline__ void inverse(Z* v, const Tables& W, unsigned char* lds, bool on, const double2* weighted) {
    typedef Geo<LOGC> G;
    typedef Geo<LOGF> F;
    typedef Pos<LOGC> P;
    constexpr u32 SUB = 1u << (LOGF - LOGC);
    double* X = (double*)lds;
    fence();
    if (on) {
        if constexpr (G::R > 1) {
            across<G::R, true>(v, tid());
            settle(v);
            twiddle<true>(v, (const d2*)(lds + F::o2) + SUB * P(tid()).j2, F::R2);
            settle(v);
        }
        last16<LOGC, true>(v);
        settle(v);
        {
            const P p(tid());
            exchange<false, P::X2, P::X1>(v, X, p.x2, p.x1, true);
        }
        twiddle<true>(v, (const d2*)(lds + F::o1) + SUB * P(tid()).j1, F::S1);
        settle(v);
        dft16<true>(v);
        settle(v);
    }
    wsync();
    const Twiddle0<true, G::T, SUB> f(W.t0, weighted, on ? tid() : 0);
    {
        const P p(tid());
        exchange<true, P::X1, P::X0>(v, X, p.x1, p.x0, on);
    }
    if (on) {
        f.apply(v);
        settle(v);
        dft16<true>(v);
        settle(v);
    }
}

// ---- Carries over the workgroup: 8 limb sums per thread, thread 0 lowest ----------------------
// Sums (biased: not negative) that stay below 2^64 with a carry of 32 bits added; limbs in l. Returns the
// carry out. `sc`: 32 words of scratch, another for the next call.
template <u32 WAVES> __device__ __forceinline__ u32 bcarry(const u64* v, u32* l, u32* sc, u32 t) {
    const u32 lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    u32 c = 0;
#pragma unroll
    for (u32 i = 0; i < 8; i++) {
        const u64 s = v[i] + c;
        l[i] = (u32)s;
        c = (u32)(s >> 32);
    }
    const u32 C = c;
    if (lane == 63) sc[w] = C;
    u32 in = (u32)__builtin_amdgcn_update_dpp(0, (int)C, 0x138, 0xf, 0xf, false);  // wave_shr:1
    __syncthreads();
    if (lane == 0) in = w ? sc[w - 1] : 0;
    u64 s = (u64)l[0] + in;
    l[0] = (u32)s;
    u32 c1 = (u32)(s >> 32);
    u32 ones = l[0];
#pragma unroll
    for (u32 i = 1; i < 8; i++) {
        s = (u64)l[i] + c1;
        l[i] = (u32)s;
        c1 = (u32)(s >> 32);
        ones &= l[i];
    }
    const u64 g = __ballot(c1 != 0), p = __ballot(ones == 0xffffffffu);
    const u64 a = g | p, sum = a + g;
    if (lane == 0) sc[16 + w] = (sum < a ? 1u : 0u) | (sum + 1 <= a && a ? 2u : 0u);
    __syncthreads();
    // Waves: generate (bit 0), and carry out when a carry comes in (bit 1).
    const u32 f = lane < WAVES ? sc[16 + lane] : 0;
    const u32 gm = (u32)__ballot(f & 1), pm = (u32)__ballot(f & 2) | gm;
    const u32 cw = (pm + gm) ^ pm ^ gm;  // bit w: a carry into wave w
    const u32 out = sc[WAVES - 1] + ((cw >> WAVES) & 1);
    const u64 cm = (a + g + ((cw >> w) & 1)) ^ a ^ g;
    if (cm) {
        c1 = (u32)(cm >> lane) & 1;
#pragma unroll
        for (u32 i = 0; i < 8; i++) {
            s = (u64)l[i] + c1;
            l[i] = (u32)s;
            c1 = (u32)(s >> 32);
        }
    }
    return out;
}

// One thread adds v to a biased number of k words, modulo R + 1 (a carry out of the top, of weight R,
// comes back in as its negative). Stops at the first word that takes no carry: usually the first.
__device__ inline void add_small(u32* w, u32 k, i64 v) {
    while (v != 0) {
        for (u32 q = 0; q < k && v != 0; q++) {
            const i64 s = (i64)w[q] + v;
            w[q] = (u32)s;
            v = s >> 32;
        }
        v = -v;
    }
}
// Sign of the biased number of k words (multiples of 64): 1 below 0x8000..8000, 0 above, 2 there. One
// whole wave; its first 64 words from the top almost always tell.
template <u32 BIASED = SGN> __device__ inline u32 sign_of(const u32* w, u32 k) {
    const u32 lane = threadIdx.x & 63;
    for (u32 q = k; q != 0; q -= 64) {
        const u32 v = w[q - 64 + lane];
        const u64 lt = __ballot(v < BIASED), gt = __ballot(v > BIASED);
        if (lt | gt) return lt > gt;
    }
    return 2;
}

// x from the K words w (biased, carried; `top` stands above them), its flag in the first wave's ex, and the
// overflow check: nonzero in some thread of the NT. Tl: T's biased halves, et what stands above them.
template <u32 BIASED, u32 NT>
__device__ __forceinline__ u32 fix_number(u32* w, u32 K, u32 top, u32 et, const u32* Tl, u32* flag, u32& ex) {
    u32 bad = 0;
    const u32 t = tid();
    if (t < 64) {
        if (t == 0) add_small(w, K, -(i64)(int)top);
        wsync();
        // X'' = words - bias is x, or x - (R + 1) where x > R / 2. A top word of zero leaves that open
        // only if T / R is in the upper half itself (its top word is read then: x below R / 2
        // is short of its bucket and has zeros there in every step).
        u32 neg = w[K - 1] < BIASED;
        if (w[K - 1] == BIASED && (et || Tl[2 * K - 1] - BIASED >= 0x40000000u)) neg = sign_of<BIASED>(w, K) & 1;
        ex = neg;
        if (neg) {
            if (t == 0) add_small(w, K, 1);
            wsync();
            if (sign_of<BIASED>(w, K) == 2) bad = 1;  // x = R stands as digits 0 and ex = 1
        }
        if (t == 0) flag[1] = neg;
    }
    __syncthreads();
    // x is T / R + m N / R (within 1) with m N / R < N, or that less R + 1 if it passed R: the
    // top limbs tell.
    if (t == NT - 1) {
        const i64 d = (i64)w[K - 1] - (i64)Tl[2 * K - 1] + ((i64)flag[1] << 32) - ((i64)et << 32);
        bad |= d < -4;
    }
    return bad;
}

// ---- The step -----------------------------------------------------------------------------------
template <u32 LOGC> struct Slot {
    typedef Geo<LOGC> G;
    static constexpr u32 C = G::C, T = G::T, k = G::k, H = C / 2;
    static constexpr u32 XT = T + T / 16;  // spaced(T, 1)
    const Args& A;
    unsigned char* const lds;
    double* X;   // exchange buffer; the digits' words and the limb sums' staging too
    u32* sc;     // carry scratch, three sets
    u32* flag;
    u32 ex = 0;  // thread 0: x = digits + ex R

    __device__ __forceinline__ Slot(const Args& a, unsigned char* l)
        : A(a), lds(l), X((double*)l), sc((u32*)(l + G::osc)), flag(sc + 96) {
        // The later passes' twiddles (a barrier follows with the first digits).
        for (u32 i = threadIdx.x; i < 16 * G::S1; i += T) ((double2*)(l + G::o1))[i] = A.w.t1[i];
        for (u32 i = threadIdx.x; i < 16 * G::R2; i += T) ((double2*)(l + G::o2))[i] = A.w.t2[i];
    }
    __device__ __forceinline__ u32* words() const { return (u32*)X; }
    // Digit j of the words (limb j / 2).
    __device__ __forceinline__ double digit(u32 j) const { return (double)(int)(int16_t)(((const uint16_t*)X)[j] ^ 0x8000); }

    __device__ __forceinline__ void put(const u32* l) { put_at(words(), l); }
    __device__ __forceinline__ void put_at(u32* p, const u32* l) {
        uint4* w = (uint4*)(p + 8 * tid());
        w[0] = make_uint4(l[0], l[1], l[2], l[3]);
        w[1] = make_uint4(l[4], l[5], l[6], l[7]);
    }
    // The words' number, weighted, in pass-0 layout; top: its digit C (thread 0's only).
    __device__ __forceinline__ void load(Z* v, u32 top) {
        const u32 t = tid();
#pragma unroll
        for (u32 e = 0; e < 16; e++) {
            const double d = digit(t + T * e);
            v[e] = Z{d * wre(e), d * wim(e)};
        }
        if (t == 0) v[0].i = (double)top;
    }
    // The same at the half length: digits j and j + H.
    __device__ __forceinline__ void load_half(Z* v, bool on) {
        if (!on) return;
        const u32 t = tid();
#pragma unroll
        for (u32 e = 0; e < 16; e++) v[e] = mulw<false>(Z{digit(t + T / 2 * e), digit(t + T / 2 * e + H)}, wre(e), wim(e));
    }
    // A transform's output f (n times the coefficient, n its length), rounded, into staging.
    template <u32 N> __device__ __forceinline__ void stage(u32 x, double f) { X[x] = __builtin_fma(f, 1.0 / N, MAGIC); }
    // Limb sum i of this thread's 8, from staging: coefficients 16 t + 2 i and 16 t + 2 i + 1.
    __device__ __forceinline__ i64 sum(u32 t, u32 i) const {
        const u64* S = (const u64*)X + G::at(16 * t) + 2 * i;
        return (i64)(S[0] + (S[1] << 16) - (MAGIC_BITS + (MAGIC_BITS << 16)));
    }
    // The limb sums of c times the staged coefficients, biased, through the carry. `in`: added at
    // limb 0 (BETA, or the carry of the half below, which holds it).
    __device__ __forceinline__ u32 carry_staged(u32 c, u32 in, u32* l, u32* scratch) {
        u64 s[8];
        const u32 t = tid();
#pragma unroll
        for (u32 i = 0; i < 8; i++) {
            i64 q = sum(t, i);
            if (c != 1) q *= (i64)c;
            s[i] = (u64)q + BIAS + SGN;
        }
        if (t == 0) s[0] += in;
        return bcarry<G::waves>(s, l, scratch, t);
    }

    // Whether T' (its biased halves at Tl) is negative; rare. Workgroup-uniform.
    __device__ __forceinline__ u32 t_negative(const u32* Tl, u32 K) {
        __syncthreads();  // every thread's halves written
        if (tid() < 64) flag[1] = sign_of(Tl, 2 * K) & 1;
        __syncthreads();
        const u32 neg = flag[1];
        __syncthreads();
        return neg;
    }

    // T = c x^2, or c x times the number of spectrum `by` (digit C of that number: ea), from the words
    // (barrier before): biased limbs of its halves to Tl (k each; each thread rereads only its
    // own), the low half in lo too. Returns what stands above T (in units of R^2, workgroup-uniform).
    __device__ __forceinline__ u32 square(u32 c, u32* lo, u32* Tl, const double2* by = nullptr, u32 ea = 1) {
        Z v[16];
        if (tid() == 0) flag[0] = ex & ea;
        load(v, ex);
        settle(v);
        __syncthreads();
        forward<LOGC, LOGC>(v, A.w, lds, true, A.w.t0);
        if (by) {
            Spectrum<T>(by, tid()).apply(v);
        } else {
#pragma unroll
            for (u32 e = 0; e < 16; e++) v[e] = Z{(v[e].r + v[e].i) * (v[e].r - v[e].i), 2.0 * v[e].r * v[e].i};
        }
        settle(v);
        inverse<LOGC, LOGC>(v, A.w, lds, true, A.w.t0);
        __syncthreads();
        {
            const u32 x = G::at(tid());
#pragma unroll
            for (u32 e = 0; e < 16; e++) {
                const Z z = mulw<true>(v[e], wre(e), wim(e));
                stage<C>(x + XT * e, z.r);
                v[e].i = z.i;
            }
        }
        fence();
        __syncthreads();
        // The product of the digits C stands at 2 C, where X^2C = -1: c more at the bottom and the top.
        const u32 up = c * flag[0];
        const u32 mid = carry_staged(c, (u32)BETA + up, lo, sc);
        put_at(Tl, lo);
        fence();
        {
            const u32 x = G::at(tid());
#pragma unroll
            for (u32 e = 0; e < 16; e++) stage<C>(x + XT * e, v[e].i);
        }
        fence();
        __syncthreads();
        u32 hi[8];
        const u32 top = carry_staged(c, mid, hi, sc + 32);
        put_at(Tl + k, hi);
        return top - (u32)BETA + up;
    }

    __device__ __forceinline__ u32 fix_x(u32 K, u32 top, u32 et, const u32* Tl) {
        return fix_number<SGN, T>(words(), K, top, et, Tl, flag, ex);
    }

    // One step on the words; returns nonzero (in some thread) on a carry that must vanish but does not.
    __device__ __forceinline__ u32 step(u32 c, const double2* np, const double2* nh, u32* Tl, const double2* by = nullptr, u32 ea = 1) {
        u32 bad = 0, et;
        {
            u32 lo[8];
            et = square(c, lo, Tl, by, ea);
            __syncthreads();
            if (et != 0) {  // T = T' + et R^2: only T' < 0 with et = 1 stands for a number below R^2
                const u32 neg = t_negative(Tl, k);
                bad |= et != neg;
                et = neg;
            }
            put(lo);
        }
        return bad | reduce(np, nh, Tl, et);
    }
    // x = (T + m N) / R from T: its biased halves at Tl, the low one in the words too, and what stands
    // above them: 1 for T' < 0, else 0.
    __device__ __forceinline__ u32 reduce(const double2* np, const double2* nh, const u32* Tl, u32 et) {
        // m = (T mod R) N' mod R.
        __syncthreads();
        Z v[16];
        load(v, 0);
        settle(v);
        __syncthreads();
        forward<LOGC, LOGC>(v, A.w, lds, true, A.w.t0);
        Spectrum<T>(np, tid()).apply(v);
        settle(v);
        inverse<LOGC, LOGC>(v, A.w, lds, true, A.w.t0);
        __syncthreads();
        {
            const u32 x = G::at(tid());
#pragma unroll
            for (u32 e = 0; e < 16; e++) stage<C>(x + XT * e, __builtin_fma(v[e].r, wre(e), v[e].i * wim(e)));
        }
        fence();
        __syncthreads();
        u32 l[8];
        carry_staged(1, (u32)BETA, l, sc + 64);
        put(l);
        __syncthreads();
        if (tid() < 64 && sign_of(words(), k) == 1 && tid() == 0) add_small(words(), k, -1);  // m = m' + R = m' - 1
        __syncthreads();
        // V = m N mod (R + 1).
        const bool on = __builtin_amdgcn_readfirstlane(tid()) < T / 2;
        load_half(v, on);
        settle(v);
        __syncthreads();
        forward<LOGC, LOGC - 1>(v, A.w, lds, on, A.w.t0);
        if (on) Spectrum<T / 2>(nh, tid()).apply(v);
        settle(v);
        inverse<LOGC, LOGC - 1>(v, A.w, lds, on, A.w.t0);
        __syncthreads();
        if (on) {
            const u32 x = G::at(tid());
#pragma unroll
            for (u32 e = 0; e < 16; e++) {
                const Z z = mulw<true>(v[e], wre(e), wim(e));
                stage<H>(x + XT / 2 * e, z.r);
                stage<H>(x + XT / 2 * e + H + H / 16, z.i);
            }
        }
        fence();
        __syncthreads();
        // x = floor(T / R) - (T mod R) - V (mod R + 1).
        u32 top;
        {
            u64 s[8];
            const u32 t = tid();
            const u32* p = Tl + 8 * t;
#pragma unroll
            for (u32 i = 0; i < 8; i++) s[i] = (u64)((i64)p[k + i] - (i64)p[i] - sum(t, i)) + BIAS + SGN;
            if (t == 0) s[0] += BETA - et;
            top = bcarry<G::waves>(s, l, sc, t) - (u32)BETA;
        }
        put(l);
        __syncthreads();
        return fix_x(k, top, et, Tl);
    }

    // k limbs as digits into the words (barriers on both sides); returns the flag e (value =
    // digits + e R) in every thread.
    __device__ __forceinline__ u32 digits_in(const u32* src) {
        u64 s[8];
        u32 l[8];
        const u32 t = tid();
#pragma unroll
        for (u32 i = 0; i < 8; i++) s[i] = (u64)src[8 * t + i] + SGN;
        const u32 e = bcarry<G::waves>(s, l, sc + 64, t);
        __syncthreads();
        put(l);
        __syncthreads();
        return e;
    }
    // Biased limbs less the bias (in: 1 at the bottom, or the carry of the half below).
    __device__ __forceinline__ u32 unbias(u32* l, u32 in, u32* scratch) {
        u64 s[8];
        const u32 t = tid();
#pragma unroll
        for (u32 i = 0; i < 8; i++) s[i] = (u64)l[i] + (0xffffffffu - SGN);
        if (t == 0) s[0] += in;
        return bcarry<G::waves>(s, l, scratch, t);
    }
};

// Up to `bits` steps on slot `slot` (reference: `steps`, kernels/src/lib.rs:883-927). BARE runs the
// squaring alone, leaves x unchanged and writes T to A.lim (lib.rs:949-961).
template <u32 LOGC, bool BARE> __device__ __forceinline__ void steps(const Args& A, u32 slot, u32 bits, unsigned char* lds) {
    typedef Slot<LOGC> S;
    constexpr u32 k = S::k;
    S s(A, lds);
    u32* x = A.x + (size_t)slot * k;
    const u32* ex = A.exp + (size_t)slot * A.ew;
    const double2* np = A.np + (size_t)slot * S::C;
    const double2* nh = A.n + (size_t)slot * S::H;
    u32* Tl = A.lim + (size_t)slot * 3 * k;
    const u32 nb = A.nbits[slot];
    u32 pos = A.pos[slot], bad = 0;
    const u32 first = pos;
    if (!BARE) s.ex = s.digits_in(x);
    for (u32 it = 0; it < bits && pos < nb; it++, pos++) {
        const u32 c = (ex[pos >> 5] >> (31 - (pos & 31))) & 1 ? A.base : 1;
        if constexpr (BARE) {
            s.ex = s.digits_in(x);
            u32 lo[8], hi[8];
            const u32 e = s.square(c, lo, Tl);
            __syncthreads();
#pragma unroll
            for (u32 i = 0; i < 8; i++) hi[i] = Tl[k + 8 * tid() + i];
            const u32 mid = s.unbias(lo, 1, s.sc + 64);
            const u32 top = s.unbias(hi, mid, s.sc);
            bad |= top + e != 1;  // T = limbs + (top - 1 + e) R^2
            s.put_at(Tl, lo);
            s.put_at(Tl + k, hi);
            __syncthreads();
        } else {
            bad |= s.step(c, np, nh, Tl);
        }
    }
    const u32 t = tid();
    if (!BARE && pos != first) {
        u32 l[8];
        const u32* w = s.words() + 8 * t;
#pragma unroll
        for (u32 i = 0; i < 8; i++) l[i] = w[i];
        s.unbias(l, 1, s.sc + 64);
#pragma unroll
        for (u32 i = 0; i < 8; i++) x[8 * t + i] = l[i];
    }
    if (t == 0) A.pos[slot] = pos;
    if (bad) A.err[slot] = 1;
}

// x[out] <- x[a] x[b] R^-1 with out's modulus (reference: `mul_slots`, lib.rs:963-988); `spec`: scratch
// for the spectrum of x[a] (2k elements, each thread reads back its own) and T (2k limbs).
template <u32 LOGC> __device__ __forceinline__ void product(const Args& A, u32 out, u32 a, u32 b, double2* spec, unsigned char* lds) {
    typedef Slot<LOGC> S;
    constexpr u32 k = S::k, T = S::T;
    S s(A, lds);
    const u32 ea = s.digits_in(A.x + (size_t)a * k);
    {
        Z v[16];
        s.load(v, ea);
        settle(v);
        __syncthreads();
        forward<LOGC, LOGC>(v, A.w, lds, true, A.w.t0);
        const u32 t = tid();
#pragma unroll
        for (u32 e = 0; e < 16; e++) spec[T * e + t] = make_double2(v[e].r, v[e].i);
        __syncthreads();
    }
    s.ex = s.digits_in(A.x + (size_t)b * k);
    const u32 bad = s.step(1, A.np + (size_t)out * S::C, A.n + (size_t)out * S::H, (u32*)(spec + 2 * k), spec, ea);
    u32 l[8];
    const u32* w = s.words() + 8 * tid();
#pragma unroll
    for (u32 i = 0; i < 8; i++) l[i] = w[i];
    s.unbias(l, 1, s.sc + 64);
    s.put_at(A.x + (size_t)out * k, l);
    if (bad) A.err[out] = 1;
}

// x[slot] R^-1 mod N to `out` (k limbs; N itself may stand for 0): the reduction of T = x, kept at Tl (2k
// limbs). For any x below R: (x + m N) / R < N + 1.
template <u32 LOGC> __device__ __forceinline__ void plain(const Args& A, u32 slot, u32* out, u32* Tl, unsigned char* lds) {
    typedef Slot<LOGC> S;
    constexpr u32 k = S::k;
    S s(A, lds);
    const u32 e = s.digits_in(A.x + (size_t)slot * k), t = tid();
    u32 l[8], hi[8];
    const u32* w = s.words() + 8 * t;
#pragma unroll
    for (u32 i = 0; i < 8; i++) {
        l[i] = w[i];
        hi[i] = SGN + (t == 0 && i == 0 ? e : 0);
    }
    s.put_at(Tl, l);
    s.put_at(Tl + k, hi);
    s.reduce(A.np + (size_t)slot * S::C, A.n + (size_t)slot * S::H, Tl, 0);
    w = s.words() + 8 * tid();
#pragma unroll
    for (u32 i = 0; i < 8; i++) l[i] = w[i];
    s.unbias(l, 1, s.sc + 64);
    s.put_at(out, l);
}

// The spectra of N' and N of one slot from their limbs (k each).
template <u32 LOGC>
__device__ __forceinline__ void constants(const Args& A, const u32* npl, const u32* nl, double2* np, double2* nh, unsigned char* lds) {
    typedef Slot<LOGC> S;
    constexpr u32 T = S::T, k = S::k;
    S s(A, lds);
    Z v[16];
    s.digits_in(npl);
    s.load(v, 0);
    fence();
    __syncthreads();
    forward<LOGC, LOGC>(v, A.w, lds, true, A.w.t0);
    const u32 t = tid();
#pragma unroll
    for (u32 e = 0; e < 16; e++) np[T * e + t] = make_double2(v[e].r, v[e].i);
    __syncthreads();
    const u32 en = s.digits_in(nl);
    if (t == 0 && en) add_small(s.words(), k, -1);
    __syncthreads();
    const bool on = __builtin_amdgcn_readfirstlane(tid()) < T / 2;
    s.load_half(v, on);
    fence();
    __syncthreads();
    forward<LOGC, LOGC - 1>(v, A.w, lds, on, A.w.t0);
    if (on)
#pragma unroll
        for (u32 e = 0; e < 16; e++) nh[T / 2 * e + t] = make_double2(v[e].r, v[e].i);
}

// ---- k = 16,384 (L = 32,768): the product in two parts --------------------------------------------
// 32,768 complex elements would take every register of a CU. But X^C - i (C = 32,768) is (X^H - z)
// (X^H + z), H = C / 2, z = exp(i pi / 4): the product modulo each factor is a weighted transform of
// length H of a_j + z a_(j+H), or a_j - z a_(j+H) (weights exp(i pi j / 4H) and exp(5 i pi j / 4H)), and from
// the two results A and B the coefficients are (A + B) / 2 and (A - B) / 2z. The parts run one
// after the other on the length-16,384 machinery; the digits are kept packed and A as it is in the
// slot's HBM scratch, each thread reading back only what it wrote. The last product has length H itself.
// Coefficients are carried a quarter (8,192 limbs) at a time, what the staging buffer holds.
//
// The bound on the error is closest here, so counted in full (u = 2^-53; a complex product by a table
// element or constant 3 u, with fused multiply-adds): a radix-16 pass 4 u and one inner rotation
// 3 u, the four twiddle factors 12 u, radix 4 across lanes 2 u, weights 3 u; 38 u a transform, 3 u more
// for the split, 4 u for the combination: 41 + 41 + 3 + 42 = 127 u, and C 2^30 127 2^-53 = 0.496.
struct SplitSlot : Slot<14> {
    typedef Slot<14> B;
    static constexpr u32 H = C, K = 2 * k;  // limbs: K; `k` is half of them

    __device__ __forceinline__ SplitSlot(const Args& a, unsigned char* l) : B(a, l) {}

    // The element weights of a part (wave-uniform loads).
    __device__ __forceinline__ const double2* weights(u32 p) const {
        u64 w = (u64)(A.w.ts + 8 * T + 16 * p);
        asm volatile("" : "+s"(w));
        return (const double2*)w;
    }
    // Part p of the words' number, weighted; its digits go to dig in part 0 and come from it in part 1.
    __device__ __forceinline__ void load_part(Z* v, u32 p, u32 top, u32* dig) {
        const double2* w = weights(p);
        const double s = p ? -RH : RH;
        const u32 t = tid();
#pragma unroll
        for (u32 e = 0; e < 16; e++) {
            u32 d;
            if (p == 0) {
                const u16* W = (const u16*)X;
                d = (u32)W[t + T * e] | (u32)W[t + T * e + H] << 16;
                d ^= SGN;
                dig[T * e + t] = d;
            } else
                d = dig[T * e + t];
            const double lo = (double)(int)(int16_t)d, hi = (double)((int)d >> 16);
            double zr = __builtin_fma(hi, s, lo);
            double zi = hi * s;
            if (e == 0 && t == 0) zi += (double)top;
            const double2 we = w[e];
            v[e] = mulw<false>(Z{zr, zi}, we.x, we.y);
            if (e % 4 == 3) fence();
        }
    }
    // A product by both parts, from the words (barrier before): the square, or times the spectrum np.
    // A is left in `part`, B in v.
    __device__ __forceinline__ void parts(Z* v, u32 top, const double2* np, double2* part, u32* dig) {
        u32 p = 0;
#pragma clang loop unroll(disable)
        do {
            load_part(v, p, top, dig);
            settle(v);
            __syncthreads();
            forward<14, 14>(v, A.w, lds, true, A.w.ts + 4 * T * p);
            if (np) {
                Spectrum<T>(np + H * p, tid()).apply(v);
            } else {
#pragma unroll
                for (u32 e = 0; e < 16; e++) v[e] = Z{(v[e].r + v[e].i) * (v[e].r - v[e].i), 2.0 * v[e].r * v[e].i};
            }
            settle(v);
            inverse<14, 14>(v, A.w, lds, true, A.w.ts + 4 * T * p);
            const double2* w = weights(p);
            const u32 t = tid();
#pragma unroll
            for (u32 e = 0; e < 16; e++) {
                const double2 we = w[e];
                v[e] = mulw<true>(v[e], we.x, we.y);
                if (p == 0) part[T * e + t] = make_double2(v[e].r, v[e].i);
                if (e % 4 == 3) fence();
            }
            settle(v);
        } while (++p < 2);
    }
    // Quarter q of the coefficients of parts() into staging (barriers around it are the caller's).
    __device__ __forceinline__ void stage_quarter(const Z* v, u32 q, const double2* part) {
        const u32 t = tid(), x = G::at(t);
#pragma unroll
        for (u32 e = 0; e < 16; e++) {
            const double2 a = part[T * e + t];
            const double dr = a.x - v[e].r, di = a.y - v[e].i;
            const double f = q == 0 ? a.x + v[e].r : q == 1 ? RH * (dr + di) : q == 2 ? a.y + v[e].i : RH * (di - dr);
            stage<2 * H>(x + XT * e, f);
            if (e % 4 == 3) fence();
        }
    }

    // T = c x^2, or by the spectrum `by`, as Slot::square: biased limbs to Tl (2K; each thread rereads
    // only its own). Returns what stands above T.
    __device__ __forceinline__ u32 square(u32 c, u32* Tl, double2* part, u32* dig, const double2* by = nullptr, u32 ea = 1) {
        Z v[16];
        if (tid() == 0) flag[0] = ex & ea;
        parts(v, ex, by, part, dig);
        const u32 up = c * flag[0];  // as in Slot::square
        u32 in = (u32)BETA + up, q = 0;
#pragma clang loop unroll(disable)
        do {
            __syncthreads();
            stage_quarter(v, q, part);
            fence();
            __syncthreads();
            u32 l[8];
            in = carry_staged(c, in, l, sc);
            put_at(Tl + k * q, l);
        } while (++q < 4);
        return in - (u32)BETA + up;
    }
    // The low half of T into the words.
    __device__ __forceinline__ void put_low(const u32* Tl) {
#pragma unroll
        for (u32 h = 0; h < 2; h++) {
            u32 l[8];
            const u32* p = Tl + k * h + 8 * tid();
#pragma unroll
            for (u32 i = 0; i < 8; i++) l[i] = p[i];
            put_at(words() + k * h, l);
        }
    }

    __device__ __forceinline__ u32 step(u32 c, const double2* np, const double2* nh, u32* Tl, double2* part, u32* dig,
                                        const double2* by = nullptr, u32 ea = 1) {
        u32 bad = 0, et = square(c, Tl, part, dig, by, ea);
        __syncthreads();
        if (et != 0) {  // as in Slot::step
            const u32 neg = t_negative(Tl, K);
            bad |= et != neg;
            et = neg;
        }
        put_low(Tl);
        return bad | reduce(np, nh, Tl, et, part, dig);
    }
    __device__ __forceinline__ u32 reduce(const double2* np, const double2* nh, const u32* Tl, u32 et, double2* part, u32* dig) {
        __syncthreads();
        Z v[16];
        parts(v, 0, np, part, dig);
        u32 l0[8], l1[8];
        __syncthreads();
        stage_quarter(v, 0, part);
        fence();
        __syncthreads();
        const u32 mid = carry_staged(1, (u32)BETA, l0, sc + 64);
        __syncthreads();
        stage_quarter(v, 1, part);
        fence();
        __syncthreads();
        carry_staged(1, mid, l1, sc + 32);
        __syncthreads();
        put_at(words(), l0);
        put_at(words() + k, l1);
        __syncthreads();
        if (tid() < 64 && sign_of(words(), K) == 1 && tid() == 0) add_small(words(), K, -1);
        __syncthreads();
        // V = m N mod (R + 1).
        {
            const u32 t = tid();
#pragma unroll
            for (u32 e = 0; e < 16; e++) v[e] = mulw<false>(Z{digit(t + T * e), digit(t + T * e + H)}, wre(e), wim(e));
        }
        settle(v);
        __syncthreads();
        forward<14, 14>(v, A.w, lds, true, A.w.t0);
        Spectrum<T>(nh, tid()).apply(v);
        settle(v);
        inverse<14, 14>(v, A.w, lds, true, A.w.t0);
#pragma unroll
        for (u32 e = 0; e < 16; e++) v[e] = mulw<true>(v[e], wre(e), wim(e));
        settle(v);
        u32 in = (u32)BETA - et;
#pragma unroll
        for (u32 h = 0; h < 2; h++) {
            __syncthreads();
            const u32 x = G::at(tid());
#pragma unroll
            for (u32 e = 0; e < 16; e++) stage<H>(x + XT * e, h ? v[e].i : v[e].r);
            fence();
            __syncthreads();
            u64 s[8];
            const u32 t = tid();
            const u32* p = Tl + k * h + 8 * t;
#pragma unroll
            for (u32 i = 0; i < 8; i++) s[i] = (u64)((i64)p[K + i] - (i64)p[i] - sum(t, i)) + BIAS + SGN;
            if (t == 0) s[0] += in;
            in = bcarry<G::waves>(s, h ? l1 : l0, sc + 32 * h, t);
        }
        __syncthreads();
        put_at(words(), l0);
        put_at(words() + k, l1);
        __syncthreads();
        return fix_x(K, in - (u32)BETA, et, Tl);
    }

    __device__ __forceinline__ u32 digits_in(const u32* src) {
        u64 s[8];
        u32 l0[8], l1[8];
        const u32 t = tid();
#pragma unroll
        for (u32 i = 0; i < 8; i++) s[i] = (u64)src[8 * t + i] + SGN;
        const u32 mid = bcarry<G::waves>(s, l0, sc + 64, t);
#pragma unroll
        for (u32 i = 0; i < 8; i++) s[i] = (u64)src[k + 8 * t + i] + SGN;
        if (t == 0) s[0] += mid;
        const u32 e = bcarry<G::waves>(s, l1, sc + 32, t);
        __syncthreads();
        put_at(words(), l0);
        put_at(words() + k, l1);
        __syncthreads();
        return e;
    }
    // The number of `quarters` times 8,192 biased limbs at src, without its bias, to dst; returns the carry.
    __device__ __forceinline__ u32 unbias_all(const u32* src, u32* dst, u32 quarters) {
        u32 in = 1;
#pragma clang loop unroll(disable)
        for (u32 q = 0; q < quarters; q++) {
            u32 l[8];
            const u32* p = src + k * q + 8 * tid();
#pragma unroll
            for (u32 i = 0; i < 8; i++) l[i] = p[i];
            __syncthreads();
            in = unbias(l, in, sc + 64);
            put_at(dst + k * q, l);
        }
        return in;
    }
};

template <bool BARE> __device__ __forceinline__ void steps_split(const Args& A, u32 slot, u32 bits, unsigned char* lds) {
    typedef SplitSlot S;
    constexpr u32 K = S::K;
    S s(A, lds);
    u32* x = A.x + (size_t)slot * K;
    const u32* ex = A.exp + (size_t)slot * A.ew;
    const double2* np = A.np + (size_t)slot * 2 * S::H;
    const double2* nh = A.n + (size_t)slot * S::H;
    double2* part = A.part + (size_t)slot * S::H;
    u32* dig = A.dig + (size_t)slot * S::H;
    u32* Tl = A.lim + (size_t)slot * 3 * K;
    const u32 nb = A.nbits[slot];
    u32 pos = A.pos[slot], bad = 0;
    const u32 first = pos;
    if (!BARE) s.ex = s.digits_in(x);
    for (u32 it = 0; it < bits && pos < nb; it++, pos++) {
        const u32 c = (ex[pos >> 5] >> (31 - (pos & 31))) & 1 ? A.base : 1;
        if constexpr (BARE) {
            s.ex = s.digits_in(x);
            const u32 e = s.square(c, Tl, part, dig);
            const u32 top = s.unbias_all(Tl, Tl, 4);
            bad |= top + e != 1;  // T = limbs + (top - 1 + e) R^2
            __syncthreads();
        } else {
            bad |= s.step(c, np, nh, Tl, part, dig);
        }
    }
    if (!BARE && pos != first) s.unbias_all(s.words(), x, 2);
    if (tid() == 0) A.pos[slot] = pos;
    if (bad) A.err[slot] = 1;
}

__device__ __forceinline__ void product_split(const Args& A, u32 out, u32 a, u32 b, double2* spec, unsigned char* lds) {
    typedef SplitSlot S;
    constexpr u32 K = S::K, H = S::H, T = S::T;
    S s(A, lds);
    u32* dig = A.dig + (size_t)out * H;
    const u32 ea = s.digits_in(A.x + (size_t)a * K);
    u32 p = 0;
#pragma clang loop unroll(disable)
    do {
        Z v[16];
        s.load_part(v, p, ea, dig);
        settle(v);
        __syncthreads();
        forward<14, 14>(v, A.w, lds, true, A.w.ts + 4 * T * p);
        const u32 t = tid();
#pragma unroll
        for (u32 e = 0; e < 16; e++) spec[H * p + T * e + t] = make_double2(v[e].r, v[e].i);
        __syncthreads();
    } while (++p < 2);
    s.ex = s.digits_in(A.x + (size_t)b * K);
    const u32 bad = s.step(1, A.np + (size_t)out * 2 * H, A.n + (size_t)out * H, (u32*)(spec + 2 * K), A.part + (size_t)out * H, dig, spec, ea);
    s.unbias_all(s.words(), A.x + (size_t)out * K, 2);
    if (bad) A.err[out] = 1;
}

__device__ __forceinline__ void plain_split(const Args& A, u32 slot, u32* out, u32* Tl, unsigned char* lds) {
    typedef SplitSlot S;
    constexpr u32 k = S::k, K = S::K;
    S s(A, lds);
    const u32 e = s.digits_in(A.x + (size_t)slot * K), t = tid();
#pragma unroll
    for (u32 h = 0; h < 2; h++) {
        u32 l[8], hi[8];
        const u32* w = s.words() + k * h + 8 * t;
#pragma unroll
        for (u32 i = 0; i < 8; i++) {
            l[i] = w[i];
            hi[i] = SGN + (h == 0 && t == 0 && i == 0 ? e : 0);
        }
        s.put_at(Tl + k * h, l);
        s.put_at(Tl + K + k * h, hi);
    }
    s.reduce(A.np + (size_t)slot * 2 * S::H, A.n + (size_t)slot * S::H, Tl, 0, A.part + (size_t)slot * S::H, A.dig + (size_t)slot * S::H);
    s.unbias_all(s.words(), out, 2);
}

// The spectra of N' (both parts) and N of one slot from their limbs.
__device__ __forceinline__ void constants_split(const Args& A, const u32* npl, const u32* nl, double2* np, double2* nh, u32* dig,
                                                unsigned char* lds) {
    typedef SplitSlot S;
    constexpr u32 T = S::T, K = S::K, H = S::H;
    S s(A, lds);
    Z v[16];
    s.digits_in(npl);
    u32 p = 0;
#pragma clang loop unroll(disable)
    do {
        s.load_part(v, p, 0, dig);
        settle(v);
        __syncthreads();
        forward<14, 14>(v, A.w, lds, true, A.w.ts + 4 * T * p);
        const u32 t = tid();
#pragma unroll
        for (u32 e = 0; e < 16; e++) np[H * p + T * e + t] = make_double2(v[e].r, v[e].i);
        __syncthreads();
    } while (++p < 2);
    const u32 en = s.digits_in(nl);
    if (tid() == 0 && en) add_small(s.words(), K, -1);
    __syncthreads();
    const u32 t = tid();
#pragma unroll
    for (u32 e = 0; e < 16; e++) v[e] = mulw<false>(Z{s.digit(t + T * e), s.digit(t + T * e + H)}, wre(e), wim(e));
    settle(v);
    __syncthreads();
    forward<14, 14>(v, A.w, lds, true, A.w.t0);
#pragma unroll
    for (u32 e = 0; e < 16; e++) nh[T * e + t] = make_double2(v[e].r, v[e].i);
}

// Host side (mm_fd.hip).
// Whether a batch of k limbs and base c can run on this path.
bool fits(u32 k, u32 base);
// exp(2 pi i num / den), den a power of two >= 8.
double2 unit(u64 num, u64 den);
// The tables of complex length C, back to back: 7 C/16, C/16, C/256, and for the split length 2C
// C/2 and 32 elements.
void make_tables(u32 C, double2* out);
inline size_t table_elems(u32 C) { return C + C / 256 + 32; }
inline Tables tables_at(const double2* p, u32 C) { return Tables{p, p + 7 * (C / 16), p + C / 2, p + C / 2 + C / 256}; }
// Transform length of a batch of k limbs: 2k, or k for the one that runs in two parts.
inline u32 length(u32 k) { return k == 16384 ? k : 2 * k; }
hipError_t set_lds_limit();
hipError_t launch(const Args& A, u32 k, u32 slots, u32 bits, bool bare, hipStream_t sm);
// x[out] <- x[a] x[b] R^-1; spec: mul_elems(k) elements of scratch.
inline size_t mul_elems(u32 k) { return 2 * k + k / 2; }
hipError_t launch_mul(const Args& A, u32 k, u32 out, u32 a, u32 b, double2* spec, hipStream_t sm);
// x R^-1 mod N (or N for 0) of `count` slots from `first`: k limbs each to out; T: 2k limbs each.
hipError_t launch_plain(const Args& A, u32 k, u32 first, u32 count, u32* out, u32* T, hipStream_t sm);
// The spectra of `count` slots from their limbs (npl, nl: k words per slot).
hipError_t launch_constants(const Args& A, u32 k, u32 count, const u32* npl, const u32* nl, double2* np, double2* nh, hipStream_t sm);

}  // namespace fd
}  // namespace mm
