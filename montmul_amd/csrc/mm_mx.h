// mm_mx.h - the Montgomery step on the integer matrix cores (wraparound path, k = L/2 limbs).
//
// A residue is n = 4k signed digits in base 256 (-128 .. 127), so a product is a convolution of
// byte strings, and a convolution is a matrix product: output digit c = 32 i1 + i0 is
//     sum_j a[i0 - j] b[32 i1 + j],
// row i0 of a 32-row Toeplitz matrix of a times column i1 of the matrix whose columns are the
// 32-digit blocks of b. v_mfma_i32_32x32x32_i8 takes 32 values of j at a time: the a operand at
// step kappa (j = -32 kappa .. -32 kappa + 31) is the Toeplitz block a[32 kappa + i0 - j'], the b
// operand is the 32 consecutive blocks of b from i1 - kappa, which the LDS holds in two planes (the
// blocks' first and second 16 bytes), each lane's 16 bytes next to its neighbour's: with whole blocks
// 32 bytes apart every read took two cycles for one. Sums are exact in 32 bits (n 2^14 <= 2^26).
//
// One wave steps one slot: no barrier anywhere. A step (R = 2^(32k) = 256^n) is
//     T = c x^2                              2n columns
//     m = (T mod R) N' mod R                 the n low columns
//     x = (T + m N) / R                      the n high columns of m N
// The low columns of m N are not formed. Their sum L with T's low half is a multiple q R, exactly;
// the last four columns give q within 2^-13, so rounding gives q itself (columns below
// n - 4 add less than n 2^14 / 255 * 256^-4 < 2^-13 in units of R).
//
// Signed digits: value + 0x80..80, carried as an ordinary number, then each byte xor 0x80. A
// value v < R is v' + e R with v' its n signed digits and e = 1 where v' < 0; the flags e of x,
// m and N enter the products as shifted terms (e_x 2 x' R and so on), which are rare but exact.
// Columns are combined four at a time into limbs (64-bit sums), and a constant that vanishes
// modulo the top limb (BETA (2^32 - 1) on every limb, BETA more on limb 0: BETA R in total) keeps
// them nonnegative through the carry.
//
// Measured against the transform kernels it replaces by default (4,096 slots unless said):
// L = 1,024 30.6 -> 91 M squarings/s; one step of a slot among 64
// at L = 512 59 -> 5.6 us, of one among 16 at L = 256 53 -> 2.8 us (the radix-4 kernel's barriers).
// At L = 1,024 power binds as much as issue: a loop of these instructions alone on random digits
// runs at 1.64 of 2.4 GHz, this kernel with its matrix cores 60 % busy at 1.75. Before the planes, the
// fragments loaded two steps ahead and eight waves a CU it was 79 M.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mm {
namespace mx {

typedef uint32_t u32;
typedef uint64_t u64;
typedef int64_t i64;
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr u32 SGN = 0x80808080u;   // 128 in every byte
constexpr u64 BETA = 1u << 27;     // |column sums| < BETA (2^32 - 1): base * n <= 2^20
constexpr u64 BIAS = BETA * 0xffffffffull;
static_assert((u64)(1u << 20) * ((1u << 14) + 1) * 0x1010101u < BIAS, "base * n <= 2^20");

// The steps' arguments, per batch.
struct Args {
    u32* x;          // k limbs per slot
    const u32* np;   // k limbs per slot: N'
    const u32* n;    // k limbs per slot: N
    const u32* exp;  // ew words per slot, most significant bit first
    const u32* nbits;
    u32* pos;
    u32* err;
    u32* lim;        // run_bare: T (2k limbs) at 3k limbs per slot, or null
    u32 ew, base;
};

// LDS of one slot in bytes, for NB blocks of 32 digits (k = 8 NB limbs). Operands stand between
// zeros, so that fragments past either end read zeros: 64 bytes for the Toeplitz operand, 32
// blocks for the other one.
template <u32 NB> struct Lay {
    static constexpr u32 n = 32 * NB, k = 8 * NB, pad = 512;
    static constexpr u32 op = 64;                            // x, T mod R and m in turn, in order
    static constexpr u32 pl = op + n + 64;                   // two planes of x, N' and N
    static constexpr u32 plane = 4 * pad + 3 * (n / 2);
    static constexpr u32 xb = pl + pad, np = xb + n / 2 + pad, nn = np + n / 2 + pad;
    static constexpr u32 st = pl + 2 * plane;                // limb sums, 9 words of 8 bytes per 8 limbs
    static constexpr u32 bytes = st + 9 * k + (NB < 32 ? 8 : 0);  // and the limb below (high_product)
    // Limb q of the planes' operand at `area` (q = -1: zeros).
    static __device__ __forceinline__ u32 at(u32 area, int q) { return area + plane * ((u32)q >> 2 & 1) + 16 * (u32)(q >> 3) + 4 * ((u32)q & 3); }
};

// Orders a wave's LDS accesses across lanes (the LDS pipeline itself is in order per wave).
__device__ __forceinline__ void wsync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ u32 rdlane(u32 v, u32 l) { return (u32)__builtin_amdgcn_readlane((int)v, (int)l); }

// Toeplitz fragment of step kappa, before the byte selection: the five dwords that hold the
// lane's digits 32 kappa + i0 - 16 h - (0 .. 15), i0 = lane & 31, h = lane >> 5.
struct FragA { u32 d[5]; };
__device__ __forceinline__ FragA load_a(const u32* a, u32 kappa) {
    FragA f;
#pragma unroll
    for (u32 i = 0; i < 5; i++) f.d[i] = a[8 * kappa + i];
    return f;
}
__device__ __forceinline__ v4i perm_a(const FragA& f, u32 sel) {
    v4i r;
#pragma unroll
    for (u32 u = 0; u < 4; u++) r[u] = (int)__builtin_amdgcn_perm(f.d[4 - u], f.d[3 - u], sel);
    return r;
}
__device__ __forceinline__ v4i load_b(const unsigned char* b, int delta) { return *(const v4i*)(b + 16 * delta); }
// Keeps loads ahead of the matrix instructions that they are meant to overlap: the scheduler moves
// them down to their first use.
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
__device__ __forceinline__ v16i mfma(v4i a, v4i b, v16i c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }

// Per-lane constants of the fragments.
struct Lane {
    u32 id, j, h, sel;
    __device__ __forceinline__ explicit Lane(u32 lane) : id(lane), j(lane & 31), h(lane >> 5) {
        const u32 r = j & 3;
        sel = 0x01020304u + 0x01010101u * r;
    }
    __device__ __forceinline__ const u32* a(const unsigned char* p) const { return (const u32*)p + (j >> 2) - 4 * h - 4; }
    __device__ __forceinline__ const unsigned char* b(const unsigned char* p, u32 plane) const { return p + 16 * j + plane * h; }
};

// Output tiles LO .. HI-1 (1,024 digits each) of the product of two n-digit strings, n >= 1,024.
// Tile c at step kappa takes the b blocks from 32 c - kappa, so with kappa = t + 32 q and
// 32 c - kappa = 32 p - t the tiles q + p share fragments: Q + (Q + 1) loads feed Q (Q + 1) matrix
// instructions per t (Q = n / 1,024). kappa = n / 32 (rows that reach past the first block) joins
// t = 0. Loads of the next t are issued before the current one's matrix instructions.
template <u32 NB, u32 LO, u32 HI>
__device__ __forceinline__ void product(const Lane& L, const unsigned char* A, const unsigned char* B, v16i* acc) {
    constexpr int Q = NB / 32;
    const u32* pa = L.a(A);
    const unsigned char* pb = L.b(B, Lay<NB>::plane);
#pragma unroll
    for (u32 c = 0; c < HI - LO; c++)
#pragma unroll
        for (u32 i = 0; i < 16; i++) acc[c][i] = 0;
    struct Frags { FragA a[Q + 1]; v4i b[Q + 1]; };
    // Whether fragment q of a (p of b) meets any wanted tile.
    auto need = [](int q, int other_max) { return q + other_max >= (int)LO && q < (int)HI; };
    auto load = [&](Frags& F, u32 t) {
#pragma unroll
        for (int q = 0; q < Q; q++)
            if (need(q, Q)) F.a[q] = load_a(pa, t + 32 * q);
#pragma unroll
        for (int p = 0; p <= Q; p++)
            if (need(p, Q - 1)) F.b[p] = load_b(pb, 32 * p - (int)t);
    };
    // A step of the loop: the matrix instructions of t (its a fragments selected already), between
    // them the loads of t + 2 and the selection of t + 1, whose loads came a step ago.
    v4i s0[Q], s1[Q];
    auto select = [&](v4i* s, const Frags& F) {
#pragma unroll
        for (int q = 0; q < Q; q++)
            if (need(q, Q)) s[q] = perm_a(F.a[q], L.sel);
    };
    auto mult = [&](const v4i* s, const Frags& F) {
#pragma unroll
        for (int q = 0; q < Q; q++)
#pragma unroll
            for (int p = 0; p <= Q; p++)
                if (q + p >= (int)LO && q + p < (int)HI) acc[q + p - LO] = mfma(s[q], F.b[p], acc[q + p - LO]);
    };
    constexpr int MFMAS = HI - LO == 2 * Q ? Q * (Q + 1) : Q * (Q + 1) / 2;
    auto interleave = [] {
#pragma unroll
        for (int i = 0; i < MFMAS; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a matrix instruction
            __builtin_amdgcn_sched_group_barrier(0x002, (4 * Q + MFMAS - 1) / MFMAS, 0);  // selections
            __builtin_amdgcn_sched_group_barrier(0x100, (4 * Q + 1 + MFMAS - 1) / MFMAS, 0);  // LDS reads
        }
        fence();
    };
    Frags F0, F1, F2;
    // t = 0: the a fragments 0, 32, .. n / 32 against the b fragments 0, 32, .. (the one past
    // the end is zero).
#pragma unroll
    for (int q = 0; q <= Q; q++) F0.a[q] = load_a(pa, 32 * q);
#pragma unroll
    for (int p = 0; p < Q; p++) F0.b[p] = load_b(pb, 32 * p);
    load(F1, 1);
    fence();
#pragma unroll
    for (int q = 0; q <= Q; q++) {
        const v4i a = perm_a(F0.a[q], L.sel);
#pragma unroll
        for (int p = 0; p < Q; p++)
            if (q + p >= (int)LO && q + p < (int)HI) acc[q + p - LO] = mfma(a, F0.b[p], acc[q + p - LO]);
    }
    load(F2, 2);
    select(s0, F1);
    fence();
    // t = 1 .. 31, three at a time (three sets of fragments in turn; loads past t = 31 are not used, and
    // read the operands' next blocks or zeros).
#pragma nounroll
    for (u32 t = 1; t < 31; t += 3) {
        mult(s0, F1);
        load(F0, t + 2);
        select(s1, F2);
        interleave();
        mult(s1, F2);
        load(F1, t + 3);
        select(s0, F0);
        interleave();
        mult(s0, F0);
        load(F2, t + 4);
        select(s1, F1);
        interleave();
#pragma unroll
        for (int q = 0; q < Q; q++) s0[q] = s1[q];
    }
    mult(s0, F1);
}

// The same for n < 1,024: one tile, whose column 0 is b's block `shift`. Four steps' loads at a time,
// ahead of the four before them.
template <u32 NB>
__device__ __forceinline__ v16i product1(const Lane& L, const unsigned char* A, const unsigned char* B, int shift) {
    const u32* pa = L.a(A);
    const unsigned char* pb = L.b(B, Lay<NB>::plane) + 16 * shift;
    v16i acc[2];
#pragma unroll
    for (u32 i = 0; i < 16; i++) acc[0][i] = acc[1][i] = 0;
    struct Frags { FragA a[4]; v4i b[4]; };
    auto load = [&](Frags& F, u32 g) {
#pragma unroll
        for (u32 i = 0; i < 4; i++)
            if (g + i <= NB) {
                F.a[i] = load_a(pa, g + i);
                F.b[i] = load_b(pb, -(int)(g + i));
            }
        fence();
    };
    Frags F[2];
    load(F[0], 0);
#pragma unroll
    for (u32 g = 0; g <= NB; g += 4) {
        if (g + 4 <= NB) load(F[g / 4 + 1 & 1], g + 4);
#pragma unroll
        for (u32 i = 0; i < 4; i++)
            if (g + i <= NB) acc[i & 1] = mfma(perm_a(F[g / 4 & 1].a[i], L.sel), F[g / 4 & 1].b[i], acc[i & 1]);
        fence();
    }
#pragma unroll
    for (u32 i = 0; i < 16; i++) acc[0][i] += acc[1][i];
    return acc[0];
}

// Rows 4 g .. 4 g + 3 of the lane's column as a limb: three multiply-adds (the multipliers are hidden
// from the compiler, which would make shifts and adds of them).
__device__ __forceinline__ i64 limb_sum(const v16i& acc, u32 g) {
    int b8 = 1 << 8, b16 = 1 << 16, b24 = 1 << 24;
    asm("" : "+s"(b8), "+s"(b16), "+s"(b24));
    return acc[4 * g] + (i64)acc[4 * g + 1] * b8 + (i64)acc[4 * g + 2] * b16 + (i64)acc[4 * g + 3] * b24;
}
// Columns of a tile into limb sums: lane (j, h) holds rows 8 g + 4 h + (0 .. 3) of column j, the
// four digits of limb 8 j + 2 g + h of the tile. Columns from `first`, `cols` of them.
__device__ __forceinline__ void stage(i64* st, u32 tile, const v16i& acc, const Lane& L, u32 first, u32 cols) {
    const u32 j = L.j - first;
    if (j < cols) {
#pragma unroll
        for (u32 g = 0; g < 4; g++) st[288 * tile + 9 * j + 2 * g + L.h] = limb_sum(acc, g);
    }
}
template <u32 E> __device__ __forceinline__ u32 stage_pos(u32 lane, u32 i) {
    if constexpr (E >= 8)
        return (E / 8) * 9 * lane + 9 * (i / 8) + i % 8;
    else
        return E * lane + (E * lane >> 3) + i;
}

// Carries E limb sums per lane over ACT lanes (lane 0 lowest; the sums of other lanes are 0): limbs
// in l, returns the carry out. Sums < 2^60.
template <u32 E, u32 ACT> __device__ __forceinline__ u32 carry(const u64* v, u32* l, u32 lane) {
    u32 c = 0;
#pragma unroll
    for (u32 i = 0; i < E; i++) {
        const bool o = __builtin_add_overflow((u32)v[i], c, &l[i]);
        c = (u32)(v[i] >> 32) + o;
    }
    const u32 C = c;
    const u32 in = (u32)__builtin_amdgcn_update_dpp(0, (int)C, 0x138, 0xf, 0xf, false);  // wave_shr:1
    bool c1 = __builtin_add_overflow(l[0], in, &l[0]);
    u32 ones = l[0];
#pragma unroll
    for (u32 i = 1; i < E; i++) {
        c1 = __builtin_add_overflow(l[i], (u32)c1, &l[i]);
        ones &= l[i];
    }
    constexpr u64 mask = ACT == 64 ? ~0ull : (1ull << ACT) - 1;
    const u64 g = __ballot(c1) & mask, p = __ballot(ones == 0xffffffffu) & mask;
    const u64 a = g | p, sum = a + g, cm = sum ^ a ^ g;  // bit i: a carry into lane i
    const u32 out = ACT == 64 ? (sum < a ? 1u : 0u) : (u32)(cm >> ACT) & 1;
    if (cm & mask) {
        c1 = (cm >> lane) & 1;
#pragma unroll
        for (u32 i = 0; i < E; i++) c1 = __builtin_add_overflow(l[i], (u32)c1, &l[i]);
    }
    return rdlane(C, ACT - 1) + out;
}

// Sign of a number given as limbs + 0x80..80: 1 negative, 0 positive, 2 zero.
template <u32 E, u32 ACT> __device__ __forceinline__ u32 sign_of(const u32* l, u32 lane) {
    const u32 top = rdlane(l[E - 1], ACT - 1);
    if (top != SGN) return top < SGN;
    bool gt = false, lt = false;
#pragma unroll
    for (u32 i = E; i-- > 0;) {
        const bool open = !gt && !lt;
        gt |= open && l[i] > SGN;
        lt |= open && l[i] < SGN;
    }
    constexpr u64 mask = ACT == 64 ? ~0ull : (1ull << ACT) - 1;
    const u64 g = __ballot(gt) & mask, t = __ballot(lt) & mask;
    return g | t ? t > g : 2;
}

// Sum over the wave (in every lane's copy of the returned scalar).
__device__ __forceinline__ int wave_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, true);  // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, true);  // row_bcast:31
    return __builtin_amdgcn_readlane(v, 63);
}

// One slot's state on one wave.
template <u32 NB> struct Slot {
    typedef Lay<NB> Y;
    static constexpr u32 k = Y::k, Q = NB / 32;
    static constexpr u32 EK = k >= 64 ? k / 64 : 1, AK = k / EK;  // limbs per lane of a residue, and lanes
    const Lane L;
    unsigned char* const lds;
    // x = x' + ex R, N = N'' + en R over the signed digits; xb: the planes' factor of T, x itself
    // between steps.
    u32 ex = 0, exb = 0, en = 0;

    __device__ __forceinline__ Slot(u32 lane, unsigned char* base) : L(lane), lds(base) {}

    __device__ __forceinline__ u32* word(u32 off) const { return (u32*)(lds + off); }
    __device__ __forceinline__ i64* sums() const { return (i64*)(lds + Y::st); }

    // Limb i of this lane's limbs as signed digits, biased limbs l: to the Toeplitz operand, or to the
    // planes at `area`.
    __device__ __forceinline__ void put(const u32* l) {
        if (L.id < AK)
#pragma unroll
            for (u32 i = 0; i < EK; i++) word(Y::op)[EK * L.id + i] = l[i] ^ SGN;
    }
    __device__ __forceinline__ void put_planes(u32 area, const u32* l) {
        if (L.id < AK)
#pragma unroll
            for (u32 i = 0; i < EK; i++) *word(Y::at(area, EK * L.id + i)) = l[i] ^ SGN;
    }
    // The signed value of four digits.
    static __device__ __forceinline__ i64 value(u32 digits) { return (i64)(digits ^ SGN) - (i64)SGN; }

    // A residue's limbs (k words at src), biased; returns the flag.
    __device__ __forceinline__ u32 digits_in(const u32* src, u32* l) {
        u64 v[EK];
#pragma unroll
        for (u32 i = 0; i < EK; i++) v[i] = L.id < AK ? (u64)src[EK * L.id + i] + SGN : 0;
        return carry<EK, AK>(v, l, L.id);
    }
    // Factors x and xb (the same for steps), N' and N.
    __device__ void init(const u32* x, const u32* xb, const u32* np, const u32* n) {
        for (u32 o = 16 * L.id; o < Y::st; o += 1024) *(v4i*)(lds + o) = v4i{0, 0, 0, 0};
        wsync();
        u32 l[EK];
        digits_in(np, l);
        put_planes(Y::np, l);
        en = digits_in(n, l);
        put_planes(Y::nn, l);
        ex = digits_in(x, l);
        put(l);
        exb = digits_in(xb, l);
        put_planes(Y::xb, l);
        wsync();
    }
    // Biased limbs to the number itself (in: 1, or the carry of the limbs below).
    __device__ __forceinline__ u32 unbias(u32* l, u32 in) {
        u64 v[EK];
#pragma unroll
        for (u32 i = 0; i < EK; i++) v[i] = L.id < AK ? (u64)l[i] + (0xffffffffu - SGN) + (EK * L.id + i == 0 ? in : 0) : 0;
        return carry<EK, AK>(v, l, L.id);
    }
    __device__ __forceinline__ void out(u32* dst, const u32* l) {
        if (L.id < AK)
#pragma unroll
            for (u32 i = 0; i < EK; i++) dst[EK * L.id + i] = l[i];
    }
    // x's limbs, from its digits.
    __device__ void store_x(u32* x) {
        u32 l[EK];
        wsync();
#pragma unroll
        for (u32 i = 0; i < EK; i++) l[i] = L.id < AK ? word(Y::op)[EK * L.id + i] ^ SGN : 0;
        unbias(l, 1);
        out(x, l);
    }

    // The staged limb sum i of this lane (0 past the last lane).
    __device__ __forceinline__ i64 staged(u32 i) const { return L.id < AK ? sums()[stage_pos<EK>(L.id, i)] : 0; }
    // c times the staged sums, biased, through the carry; `in` joins limb 0.
    __device__ __forceinline__ u32 carry_staged(u32 c, u64 in, u32* l) {
        u64 v[EK];
#pragma unroll
        for (u32 i = 0; i < EK; i++) {
            i64 s = staged(i);
            if (c != 1) s *= (i64)c;
            v[i] = L.id < AK ? (u64)s + BIAS + SGN + (EK * L.id + i == 0 ? in : 0) : 0;
        }
        return carry<EK, AK>(v, l, L.id);
    }

    // T = c x xb as biased limbs, low and high half; returns what stands above them (in units of
    // R^2). The halves are carried one after the other, so that the sums of one half are staged.
    __device__ __forceinline__ u32 square(u32 c, u32* lo, u32* hi) {
        const unsigned char *X = lds + Y::op, *XB = lds + Y::xb;
        u32 mid;
        if constexpr (NB >= 32) {
            v16i acc[2 * Q];
            product<NB, 0, 2 * Q>(L, X, XB, acc);
#pragma unroll
            for (u32 t = 0; t < Q; t++) stage(sums(), t, acc[t], L, 0, 32);
            wsync();
            mid = carry_staged(c, BETA, lo);
            wsync();
#pragma unroll
            for (u32 t = 0; t < Q; t++) stage(sums(), t, acc[Q + t], L, 0, 32);
        } else {
            const v16i acc = product1<NB>(L, X, XB, 0);
            stage(sums(), 0, acc, L, 0, NB);
            wsync();
            mid = carry_staged(c, BETA, lo);
            wsync();
            stage(sums(), 0, acc, L, NB, NB);
        }
        wsync();
        u32 top;
        if (ex | exb) {  // + c (ex xb' R + exb x' R + ex exb R^2)
            u64 v[EK];
#pragma unroll
            for (u32 i = 0; i < EK; i++) {
                const u32 q = EK * L.id + i;
                const i64 more = (ex ? value(*word(Y::at(Y::xb, q))) : 0) + (exb ? value(word(Y::op)[q]) : 0);
                v[i] = L.id < AK ? (u64)((i64)c * (staged(i) + more)) + BIAS + SGN + (q == 0 ? mid : 0) : 0;
            }
            top = carry<EK, AK>(v, hi, L.id) + c * (ex & exb);
        } else {
            top = carry_staged(c, mid, hi);  // mid holds the low half's BETA
        }
        wsync();
        return top - (u32)BETA;
    }
    // The part of a nonzero square() that stands for a number: 1 for T' < 0 (T = T' + R^2), else 0.
    __device__ __forceinline__ u32 borrowed(const u32* lo, const u32* hi) const {
        const u32 s = sign_of<EK, AK>(hi, L.id);
        return (s == 2 ? sign_of<EK, AK>(lo, L.id) : s) & 1;
    }

    // One step; returns nonzero on a carry that must vanish but does not.
    __device__ __forceinline__ u32 step(u32 c) {
        u32 bad = 0;
        u32 l[EK], hi[EK];
        u32 et = square(c, l, hi);
        if (et) {
            const u32 neg = borrowed(l, hi);
            bad |= et != neg;
            et = neg;
        }
        return bad | reduce(l, hi, et);
    }
    // x = (T + m N) / R from T's biased halves (l, hi) and what stands above them: 1 for T' < 0, else 0.
    __device__ __forceinline__ u32 reduce(u32* l, const u32* hi, u32 et) {
        u32 bad = 0;
        // T's top limb below R, for q.
        const i64 tlow = (i64)rdlane(l[EK - 1], AK - 1) - (i64)SGN;
        put(l);
        wsync();
        // m = (T mod R) N' mod R.
        low_product();
        wsync();
        carry_staged(1, BETA, l);
        const u32 em = sign_of<EK, AK>(l, L.id) & 1;
        put(l);
        wsync();
        // The last four low columns of m N, and with T's digits there q = (L + T mod R) / R; then the
        // high columns.
        const i64 cols = high_product();
        const i64 q = (cols + tlow + (1ll << 31)) >> 32;
        // x = floor(T / R) + the high columns of m N + q + e_m N + e_N m.
        u64 v[EK];
#pragma unroll
        for (u32 i = 0; i < EK; i++) {
            const u32 j = EK * L.id + i;
            v[i] = L.id < AK ? (u64)staged(i) + BIAS + hi[i] + (j == 0 ? (u64)((i64)BETA + q) : 0) : 0;
            if (em && L.id < AK) v[i] += (u64)value(*word(Y::at(Y::nn, j)));
        }
        u32 f = et + (em & en);
        if (en) {
#pragma unroll
            for (u32 i = 0; i < EK; i++)
                if (L.id < AK) v[i] += (u64)value(word(Y::op)[EK * L.id + i]);
        }
        f += carry<EK, AK>(v, l, L.id) - (u32)BETA;
        ex = 0;
        if (f) {
            ex = sign_of<EK, AK>(l, L.id) & 1;
            bad |= f != ex;
        }
        exb = ex;
        wsync();
        put(l);
        put_planes(Y::xb, l);
        wsync();
        return bad;
    }

    __device__ __forceinline__ void low_product() {
        if constexpr (NB >= 32) {
            v16i acc[Q];
            product<NB, 0, Q>(L, lds + Y::op, lds + Y::np, acc);
#pragma unroll
            for (u32 t = 0; t < Q; t++) stage(sums(), t, acc[t], L, 0, 32);
        } else {
            stage(sums(), 0, product1<NB>(L, lds + Y::op, lds + Y::np, 0), L, 0, NB);
        }
    }
    // The high columns' limb sums of m N into staging; returns the sum of the limb below them. Below
    // n = 1,024 the tile has columns to spare and starts one of them lower (the dot products and their
    // reduction were 4 % of a step at L = 64, 2 % at 256); above, that limb's four columns come by dot
    // products.
    __device__ __forceinline__ i64 high_product() {
        if constexpr (NB >= 32) {
            int g0 = 0, g1 = 0, g2 = 0, g3 = 0;
#pragma unroll
            for (u32 r = 0; r < k / 64; r++) {
                const u32 w = 64 * r + L.id, W = k - 1 - w;
                const int md = (int)word(Y::op)[w];
                const u32 hi = *word(Y::at(Y::nn, (int)W)), lo = *word(Y::at(Y::nn, (int)W - 1));
                g0 = __builtin_amdgcn_sdot4(md, (int)__builtin_amdgcn_perm(hi, lo, 0x01020304u), g0, false);
                g1 = __builtin_amdgcn_sdot4(md, (int)__builtin_amdgcn_perm(hi, lo, 0x02030405u), g1, false);
                g2 = __builtin_amdgcn_sdot4(md, (int)__builtin_amdgcn_perm(hi, lo, 0x03040506u), g2, false);
                g3 = __builtin_amdgcn_sdot4(md, (int)__builtin_amdgcn_perm(hi, lo, 0x04050607u), g3, false);
            }
            const i64 cols = (i64)wave_sum(g0) + ((i64)wave_sum(g1) << 8) + ((i64)wave_sum(g2) << 16) + ((i64)wave_sum(g3) << 24);
            v16i acc[Q];
            product<NB, Q, 2 * Q>(L, lds + Y::op, lds + Y::nn, acc);
#pragma unroll
            for (u32 t = 0; t < Q; t++) stage(sums(), t, acc[t], L, 0, 32);
            wsync();
            return cols;
        } else {
            // Column 0 is the last below R: its limb 7 stands past the sums of the others.
            const v16i acc = product1<NB>(L, lds + Y::op, lds + Y::nn, (int)NB - 1);
            stage(sums(), 0, acc, L, 1, NB);
            if (L.id == 32) sums()[9 * NB] = limb_sum(acc, 3);
            wsync();
            return sums()[9 * NB];
        }
    }
};

// Up to `bits` steps on one slot by one wave (reference: `steps`, kernels/src/lib.rs:883-927).
// BARE runs the squaring alone, leaves x unchanged and writes T to A.lim (lib.rs:949-961).
template <u32 NB, bool BARE>
__device__ __forceinline__ void steps(const Args& A, u32 slot, u32 bits, u32 lane, unsigned char* lds) {
    typedef Slot<NB> S;
    constexpr u32 k = S::k;
    S s(lane, lds);
    const u32* x0 = A.x + (size_t)slot * k;
    s.init(x0, x0, A.np + (size_t)slot * k, A.n + (size_t)slot * k);
    const u32* ex = A.exp + (size_t)slot * A.ew;
    const u32 nb = A.nbits[slot];
    u32 pos = A.pos[slot], bad = 0;
    const u32 first = pos;
    for (u32 it = 0; it < bits && pos < nb; it++, pos++) {
        const u32 c = (ex[pos >> 5] >> (31 - (pos & 31))) & 1 ? A.base : 1;
        if constexpr (BARE) {
            u32 lo[S::EK], hi[S::EK];
            const u32 e = s.square(c, lo, hi);
            bad |= e != 0 && e != s.borrowed(lo, hi);
            if (A.lim) {
                s.unbias(hi, s.unbias(lo, 1));
                s.out(A.lim + (size_t)slot * 3 * k, lo);
                s.out(A.lim + (size_t)slot * 3 * k + k, hi);
            }
        } else {
            bad |= s.step(c);
        }
    }
    if (!BARE && pos != first) s.store_x(A.x + (size_t)slot * k);
    if (lane == 0) {
        A.pos[slot] = pos;
        if (bad) A.err[slot] = 1;
    }
}

// x[out] <- x[a] x[b] R^-1 with out's modulus, by one wave (reference: `mul_slots`, lib.rs:963-988).
template <u32 NB> __device__ __forceinline__ void product_of(const Args& A, u32 out, u32 a, u32 b, u32 lane, unsigned char* lds) {
    typedef Slot<NB> S;
    constexpr size_t k = S::k;
    S s(lane, lds);
    s.init(A.x + a * k, A.x + b * k, A.np + out * k, A.n + out * k);
    const u32 bad = s.step(1);
    s.store_x(A.x + out * k);
    if (lane == 0 && bad) A.err[out] = 1;
}

// x[slot] R^-1 mod N to `out` (k limbs; N itself may stand for 0), by one wave: the reduction of T = x. For
// any x below R: (x + m N) / R < N + 1.
template <u32 NB> __device__ __forceinline__ void plain(const Args& A, u32 slot, u32* out, u32 lane, unsigned char* lds) {
    typedef Slot<NB> S;
    constexpr u32 k = S::k;
    S s(lane, lds);
    const u32* x = A.x + (size_t)slot * k;
    s.init(x, x, A.np + (size_t)slot * k, A.n + (size_t)slot * k);
    u32 l[S::EK], hi[S::EK];
    const u32 e = s.digits_in(x, l);
#pragma unroll
    for (u32 i = 0; i < S::EK; i++) hi[i] = SGN + (S::EK * lane + i == 0 ? e : 0);
    s.reduce(l, hi, 0);
    s.store_x(out);
}

// Host side (mm_mx.hip): whether a batch can run on this path (log2 of the length L = 2k, the
// base c), and the launch of its steps, one wave per slot.
bool fits(u32 k, u32 base);
hipError_t launch(const Args& A, u32 k, u32 slots, u32 bits, bool bare, hipStream_t sm);
hipError_t launch_mul(const Args& A, u32 k, u32 out, u32 a, u32 b, hipStream_t sm);
// x R^-1 mod N (or N for 0) of `count` slots from `first`: k limbs each to out.
hipError_t launch_plain(const Args& A, u32 k, u32 first, u32 count, u32* out, hipStream_t sm);

}  // namespace mx
}  // namespace mm
