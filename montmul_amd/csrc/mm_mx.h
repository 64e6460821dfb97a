// mm_mx.h - the Montgomery step on the integer matrix cores (wraparound path, k = L/2 limbs).
//
// A residue is n = 4k signed digits in base 256 (-128 .. 127), so a product is a convolution of
// byte strings, and a convolution is a matrix product: output digit c = 32 i1 + i0 is
//     sum_j a[i0 - j] b[32 i1 + j],
// row i0 of a 32-row Toeplitz matrix of a times column i1 of the matrix whose columns are the
// 32-digit blocks of b. v_mfma_i32_32x32x32_i8 takes 32 values of j at a time: the a operand at
// step kappa (j = -32 kappa .. -32 kappa + 31) is the Toeplitz block a[32 kappa + i0 - j'], the b
// operand is the 32 consecutive blocks of b from i1 - kappa, 1 KiB contiguous in LDS. Sums are
// exact in 32 bits (n 2^14 <= 2^26).
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
// L = 1,024 30.6 -> 79 M squarings/s, 2,048 (2,048 slots) 14.4 -> 25 M; one step of a slot among 64
// at L = 512 59 -> 6.4 us, of one among 16 at L = 256 53 -> 3.5 us (the radix-4 kernel's barriers).
// At L = 1,024 LDS reads bind (77 % busy, a quarter of it bank conflicts), then the matrix cores
// (52 %, at the 1.74 GHz that dense int8 products leave of the clock).
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
// 1 KiB of zeros, so that fragments past either end read zeros.
template <u32 NB> struct Lay {
    static constexpr u32 n = 32 * NB, k = 8 * NB, pad = 1024;
    static constexpr u32 op = pad;           // x, T mod R and m in turn
    static constexpr u32 np = op + n + pad;  // N'
    static constexpr u32 nn = np + n + pad;  // N
    static constexpr u32 st = nn + n + pad;  // limb sums, 9 words of 8 bytes per 8 limbs
    static constexpr u32 th = st + 9 * k;    // floor(T / R), past the sums of k limbs
    static constexpr u32 bytes = st + 18 * k;
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
__device__ __forceinline__ v4i load_b(const unsigned char* b, int delta) { return *(const v4i*)(b + 32 * delta); }
__device__ __forceinline__ v16i mfma(v4i a, v4i b, v16i c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }

// Per-lane constants of the fragments.
struct Lane {
    u32 id, j, h, sel;
    __device__ __forceinline__ explicit Lane(u32 lane) : id(lane), j(lane & 31), h(lane >> 5) {
        const u32 r = j & 3;
        sel = 0x01020304u + 0x01010101u * r;
    }
    __device__ __forceinline__ const u32* a(const unsigned char* p) const { return (const u32*)p + (j >> 2) - 4 * h - 4 + 0; }
    __device__ __forceinline__ const unsigned char* b(const unsigned char* p) const { return p + 32 * j + 16 * h; }
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
    const unsigned char* pb = L.b(B);
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
    auto mult = [&](const Frags& F) {
#pragma unroll
        for (int q = 0; q < Q; q++)
            if (need(q, Q)) {
                const v4i a = perm_a(F.a[q], L.sel);
#pragma unroll
                for (int p = 0; p <= Q; p++)
                    if (q + p >= (int)LO && q + p < (int)HI) acc[q + p - LO] = mfma(a, F.b[p], acc[q + p - LO]);
            }
    };
    Frags F0, F1;
    // t = 0: the a fragments 0, 32, .. n / 32 against the b fragments 0, 32, .. (the one past
    // the end is zero).
#pragma unroll
    for (int q = 0; q <= Q; q++) F0.a[q] = load_a(pa, 32 * q);
#pragma unroll
    for (int p = 0; p < Q; p++) F0.b[p] = load_b(pb, 32 * p);
    load(F1, 1);
#pragma unroll
    for (int q = 0; q <= Q; q++) {
        const v4i a = perm_a(F0.a[q], L.sel);
#pragma unroll
        for (int p = 0; p < Q; p++)
            if (q + p >= (int)LO && q + p < (int)HI) acc[q + p - LO] = mfma(a, F0.b[p], acc[q + p - LO]);
    }
#pragma nounroll
    for (u32 t = 1; t < 31; t += 2) {
        load(F0, t + 1);
        mult(F1);
        load(F1, t + 2);
        mult(F0);
    }
    mult(F1);
}

// The same for n < 1,024: one tile, whose column 0 is b's block `shift`.
template <u32 NB>
__device__ __forceinline__ v16i product1(const Lane& L, const unsigned char* A, const unsigned char* B, int shift) {
    const u32* pa = L.a(A);
    const unsigned char* pb = L.b(B);
    v16i acc, acc2;
#pragma unroll
    for (u32 i = 0; i < 16; i++) acc[i] = acc2[i] = 0;
#pragma unroll
    for (u32 kappa = 0; kappa <= NB; kappa++) {
        const v4i a = perm_a(load_a(pa, kappa), L.sel);
        const v4i b = load_b(pb, shift - (int)kappa);
        if (kappa & 1)
            acc2 = mfma(a, b, acc2);
        else
            acc = mfma(a, b, acc);
    }
#pragma unroll
    for (u32 i = 0; i < 16; i++) acc[i] += acc2[i];
    return acc;
}

// Columns of a tile into limb sums: lane (j, h) holds rows 8 g + 4 h + (0 .. 3) of column j, the
// four digits of limb 8 j + 2 g + h of the tile.
__device__ __forceinline__ void stage(i64* st, u32 tile, const v16i& acc, const Lane& L, u32 cols) {
    if (L.j < cols) {
#pragma unroll
        for (u32 g = 0; g < 4; g++) {
            const i64 v = (i64)acc[4 * g] + ((i64)acc[4 * g + 1] << 8) + ((i64)acc[4 * g + 2] << 16) + ((i64)acc[4 * g + 3] << 24);
            st[288 * tile + 9 * L.j + 2 * g + L.h] = v;
        }
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
    u64 c = 0;
#pragma unroll
    for (u32 i = 0; i < E; i++) {
        const u64 s = v[i] + c;
        l[i] = (u32)s;
        c = s >> 32;
    }
    const u32 C = (u32)c;
    const u32 in = (u32)__builtin_amdgcn_update_dpp(0, (int)C, 0x138, 0xf, 0xf, false);  // wave_shr:1
    u64 s = (u64)l[0] + in;
    l[0] = (u32)s;
    u32 c1 = (u32)(s >> 32);
    bool ones = l[0] == 0xffffffffu;
#pragma unroll
    for (u32 i = 1; i < E; i++) {
        s = (u64)l[i] + c1;
        l[i] = (u32)s;
        c1 = (u32)(s >> 32);
        ones &= l[i] == 0xffffffffu;
    }
    constexpr u64 mask = ACT == 64 ? ~0ull : (1ull << ACT) - 1;
    const u64 g = __ballot(c1 != 0) & mask, p = __ballot(ones) & mask;
    const u64 a = g | p, sum = a + g, cm = sum ^ a ^ g;  // bit i: a carry into lane i
    const u32 out = ACT == 64 ? (sum < a ? 1u : 0u) : (u32)(cm >> ACT) & 1;
    if (cm & mask) {
        c1 = (u32)(cm >> lane) & 1;
#pragma unroll
        for (u32 i = 0; i < E; i++) {
            s = (u64)l[i] + c1;
            l[i] = (u32)s;
            c1 = (u32)(s >> 32);
        }
    }
    return rdlane(C, ACT - 1) + out;
}

// Whether a number given as limbs + 0x80..80 is negative.
template <u32 E, u32 ACT> __device__ __forceinline__ u32 negative(const u32* l, u32 lane) {
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
    return t > g;
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
    static constexpr u32 ET = 2 * k >= 64 ? 2 * k / 64 : 1, AT = 2 * k / ET;  // limbs per lane and lanes of T
    static constexpr u32 EK = k >= 64 ? k / 64 : 1, AK = k / EK;              // and of one residue
    const Lane L;
    unsigned char* const lds;
    u32 ex = 0, en = 0;  // x = x' + ex R, N = N'' + en R over the signed digits

    __device__ __forceinline__ Slot(u32 lane, unsigned char* base) : L(lane), lds(base) {}

    __device__ __forceinline__ u32* words(u32 off) const { return (u32*)(lds + off); }
    __device__ __forceinline__ i64* sums() const { return (i64*)(lds + Y::st); }

    // A residue's limbs (k words at src) as signed digits at `area`; returns the flag.
    __device__ __forceinline__ u32 digits_in(const u32* src, u32 area) {
        u64 v[EK];
        u32 l[EK];
#pragma unroll
        for (u32 i = 0; i < EK; i++) v[i] = L.id < AK ? (u64)src[EK * L.id + i] + SGN : 0;
        const u32 e = carry<EK, AK>(v, l, L.id);
        put(area, l);
        return e;
    }
    // Biased limbs as signed digits at `area`.
    __device__ __forceinline__ void put(u32 area, const u32* l) {
        if (L.id < AK)
#pragma unroll
            for (u32 i = 0; i < EK; i++) words(area)[EK * L.id + i] = l[i] ^ SGN;
    }
    // The signed value of limb q of the digits at `area`.
    __device__ __forceinline__ i64 limb_at(u32 area, u32 q) const { return (i64)(words(area)[q] ^ SGN) - (i64)SGN; }

    __device__ void init(const u32* x, const u32* np, const u32* n) {
        for (u32 o = 16 * L.id; o < Y::st; o += 1024) *(v4i*)(lds + o) = v4i{0, 0, 0, 0};
        wsync();
        digits_in(np, Y::np);
        en = digits_in(n, Y::nn);
        ex = digits_in(x, Y::op);
        wsync();
    }

    // x's limbs, from its digits.
    __device__ void store_x(u32* x) {
        u64 v[EK];
        u32 l[EK];
        wsync();
#pragma unroll
        for (u32 i = 0; i < EK; i++)
            v[i] = L.id < AK ? (u64)(words(Y::op)[EK * L.id + i] ^ SGN) + (0xffffffffu - SGN) + (EK * L.id + i == 0) : 0;
        carry<EK, AK>(v, l, L.id);
        if (L.id < AK)
#pragma unroll
            for (u32 i = 0; i < EK; i++) x[EK * L.id + i] = l[i];
    }

    // T = c x^2 as biased limbs, ET per lane; returns what stands above them (in units of R^2).
    __device__ __forceinline__ u32 square(u32 c, u32* l) {
        const unsigned char* X = lds + Y::op;
        if constexpr (NB >= 32) {
            v16i acc[2 * Q];
            product<NB, 0, 2 * Q>(L, X, X, acc);
#pragma unroll
            for (u32 t = 0; t < 2 * Q; t++) stage(sums(), t, acc[t], L, 32);
        } else {
            stage(sums(), 0, product1<NB>(L, X, X, 0), L, 2 * NB);
        }
        wsync();
        u64 v[ET];
#pragma unroll
        for (u32 i = 0; i < ET; i++) {
            i64 s = L.id < AT ? sums()[stage_pos<ET>(L.id, i)] : 0;
            if (c != 1) s *= (i64)c;
            v[i] = L.id < AT ? (u64)s + BIAS + SGN + (ET * L.id + i == 0 ? BETA : 0) : 0;
        }
        u32 e = 0;
        if (ex) {  // + c (2 x' R + R^2)
#pragma unroll
            for (u32 i = 0; i < ET; i++) {
                const u32 q = ET * L.id + i;
                if (L.id < AT && q >= k) v[i] += (u64)(2 * (i64)c * limb_at(Y::op, q - k));
            }
            e = c;
        }
        e += carry<ET, AT>(v, l, L.id) - (u32)BETA;
        return e;
    }

    // One step; returns nonzero on a carry that must vanish but does not.
    __device__ __forceinline__ u32 step(u32 c) {
        u32 bad = 0, lt[ET];
        u32 et = square(c, lt);
        if (et) {  // T = T' + et R^2: only T' < 0, et = 1 stands for a number below R^2
            const u32 neg = negative<ET, AT>(lt, L.id);
            bad |= et != neg;
            et = neg;
        }
        // T's top limb below R, for q.
        const i64 tlow = (i64)rdlane(lt[ET - 1], AT / 2 - 1) - (i64)SGN;
        wsync();
        if (L.id < AT / 2) {
#pragma unroll
            for (u32 i = 0; i < ET; i++) words(Y::op)[ET * L.id + i] = lt[i] ^ SGN;
        } else if (L.id < AT) {
#pragma unroll
            for (u32 i = 0; i < ET; i++) words(Y::th)[ET * L.id + i - k] = lt[i];
        }
        wsync();
        // m = (T mod R) N' mod R.
        u64 v[EK];
        u32 l[EK];
        low_product();
        wsync();
#pragma unroll
        for (u32 i = 0; i < EK; i++)
            v[i] = L.id < AK ? (u64)sums()[stage_pos<EK>(L.id, i)] + BIAS + SGN + (EK * L.id + i == 0 ? BETA : 0) : 0;
        carry<EK, AK>(v, l, L.id);
        const u32 em = negative<EK, AK>(l, L.id);
        put(Y::op, l);
        wsync();
        // The last four low columns of m N, and with T's digits there q = (L + T mod R) / R.
        int g0 = 0, g1 = 0, g2 = 0, g3 = 0;
        const u32 *mw = words(Y::op), *nw = words(Y::nn);
#pragma unroll
        for (u32 r = 0; r < (k + 63) / 64; r++) {
            const u32 w = 64 * r + L.id;
            const int md = w < k ? (int)mw[w] : 0;
            const u32 W = w < k ? k - 1 - w : 0;
            const u32 hi = nw[W], lo = nw[(int)W - 1];
            g0 = __builtin_amdgcn_sdot4(md, (int)__builtin_amdgcn_perm(hi, lo, 0x01020304u), g0, false);
            g1 = __builtin_amdgcn_sdot4(md, (int)__builtin_amdgcn_perm(hi, lo, 0x02030405u), g1, false);
            g2 = __builtin_amdgcn_sdot4(md, (int)__builtin_amdgcn_perm(hi, lo, 0x03040506u), g2, false);
            g3 = __builtin_amdgcn_sdot4(md, (int)__builtin_amdgcn_perm(hi, lo, 0x04050607u), g3, false);
        }
        const i64 cols = (i64)wave_sum(g0) + ((i64)wave_sum(g1) << 8) + ((i64)wave_sum(g2) << 16) + ((i64)wave_sum(g3) << 24);
        const i64 q = (cols + tlow + (1ll << 31)) >> 32;
        // x = floor(T / R) + the high columns of m N + q + e_m N + e_N m.
        high_product();
        wsync();
#pragma unroll
        for (u32 i = 0; i < EK; i++) {
            const u32 j = EK * L.id + i;
            v[i] = L.id < AK ? (u64)sums()[stage_pos<EK>(L.id, i)] + BIAS + words(Y::th)[j] + (j == 0 ? (u64)((i64)BETA + q) : 0) : 0;
            if (em && L.id < AK) v[i] += (u64)limb_at(Y::nn, j);
        }
        u32 f = et + (em & en);
        if (en) {
#pragma unroll
            for (u32 i = 0; i < EK; i++)
                if (L.id < AK) v[i] += (u64)limb_at(Y::op, EK * L.id + i);
        }
        f += carry<EK, AK>(v, l, L.id) - (u32)BETA;
        ex = 0;
        if (f) {
            ex = negative<EK, AK>(l, L.id);
            bad |= f != ex;
        }
        wsync();
        put(Y::op, l);
        wsync();
        return bad;
    }

    __device__ __forceinline__ void low_product() {
        if constexpr (NB >= 32) {
            v16i acc[Q];
            product<NB, 0, Q>(L, lds + Y::op, lds + Y::np, acc);
#pragma unroll
            for (u32 t = 0; t < Q; t++) stage(sums(), t, acc[t], L, 32);
        } else {
            stage(sums(), 0, product1<NB>(L, lds + Y::op, lds + Y::np, 0), L, NB);
        }
    }
    __device__ __forceinline__ void high_product() {
        if constexpr (NB >= 32) {
            v16i acc[Q];
            product<NB, Q, 2 * Q>(L, lds + Y::op, lds + Y::nn, acc);
#pragma unroll
            for (u32 t = 0; t < Q; t++) stage(sums(), t, acc[t], L, 32);
        } else {
            stage(sums(), 0, product1<NB>(L, lds + Y::op, lds + Y::nn, (int)NB), L, NB);
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
    s.init(A.x + (size_t)slot * k, A.np + (size_t)slot * k, A.n + (size_t)slot * k);
    const u32* ex = A.exp + (size_t)slot * A.ew;
    const u32 nb = A.nbits[slot];
    u32 pos = A.pos[slot], bad = 0;
    const u32 first = pos;
    for (u32 it = 0; it < bits && pos < nb; it++, pos++) {
        const u32 c = (ex[pos >> 5] >> (31 - (pos & 31))) & 1 ? A.base : 1;
        if constexpr (BARE) {
            u32 l[S::ET];
            const u32 e = s.square(c, l);
            bad |= e != 0 && e != negative<S::ET, S::AT>(l, lane);
            if (A.lim) {
                u64 v[S::ET];
#pragma unroll
                for (u32 i = 0; i < S::ET; i++) v[i] = lane < S::AT ? (u64)l[i] + (0xffffffffu - SGN) + (S::ET * lane + i == 0) : 0;
                carry<S::ET, S::AT>(v, l, lane);
                if (lane < S::AT)
#pragma unroll
                    for (u32 i = 0; i < S::ET; i++) A.lim[(size_t)slot * 3 * k + S::ET * lane + i] = l[i];
            }
            wsync();
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

// Host side (mm_mx.hip): whether a batch can run on this path (log2 of the length L = 2k, the
// base c), and the launch of its steps, one wave per slot.
bool fits(u32 k, u32 base);
hipError_t launch(const Args& A, u32 k, u32 slots, u32 bits, bool bare, hipStream_t sm);

}  // namespace mx
}  // namespace mm
