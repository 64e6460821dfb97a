// mm_fdw.h - the double-precision step at L = 65,536 (k = 32,768 limbs), several workgroups to a slot.
#pragma once

#include "mm_fd.h"

namespace mm {
namespace fdw {

using fd::Tables;
using fd::u32;
using fd::u64;
using fd::i64;

constexpr u32 K = 32768, H = 16384;

struct Args {
    Tables w;            // length H
    const double2* tw;   // the parts' weights (make_tables)
    u32* x;              // K limbs per slot
    double2* np;         // 8 H per slot: spectrum of N', part after part
    double2* n;          // 4 H per slot: spectrum of N
    const u32* exp;      // ew words per slot, most significant bit first
    const u32* nbits;
    u32* pos;
    u32* err;
    u32* lim;            // T (2K biased limbs), then m (K), per slot
    // Scratch of the slots that run together, `first` and those after it: the parts' results (8 H
    // elements), the limb sums (2K), x as biased limbs (K), x's flag and T's (2 words).
    double2* part;
    i64* sum;
    u32* dig;
    u32* fl;
    u32 ew, base, first;
};
constexpr size_t SCRATCH = 8ull * H * 16 + 2ull * K * 8 + 4ull * K + 8;  // bytes per slot
constexpr u32 GROUP = 64;                                              // slots that run together, at most

bool fits(u32 k, u32 base);
// The tables of the parts' length (fd::make_tables), then the parts' weights: TABLE elements.
constexpr size_t WEIGHTS = 48 * (H / 16) + 8 * 16 + 4 * 16 + 8 * 8 + 4 * 4;
constexpr size_t TABLE = H + H / 256 + 32 + WEIGHTS;
void make_tables(double2* out);
hipError_t set_lds_limit();
// Up to steps[g] steps on the slots [g GROUP, (g + 1) GROUP) of [0, slots).
hipError_t launch(Args A, u32 slots, const u32* steps, hipStream_t sm);
// The spectra of `count` slots from A.first on, from their limbs (npl, nl: K words per slot).
hipError_t launch_constants(Args A, u32 count, const u32* npl, const u32* nl, hipStream_t sm);

}  // namespace fdw
}  // namespace mm
