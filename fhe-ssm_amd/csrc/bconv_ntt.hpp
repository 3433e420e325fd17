// bconv_ntt.hpp -- plans and launch arguments of the BConv fused with the forward NTT's first pass (bconv_ntt.hip).
#pragma once
#include "engine.hpp"

namespace fhe {

constexpr uint32_t kMfMaxOut = 80;  // output limbs of a conversion
constexpr uint32_t kMfMaxDigits = 8;
// the quotient estimate of the reduction needs primes of at least 35 bits (its unit is 2^32)
constexpr uint64_t kMfMinQ = 1ull << 34;

constexpr uint32_t kMfNone = 1;  // unused slot

// one output of a conversion, in groups of four (the last group padded)
struct MfSlot {
    uint64_t q;
    int32_t nq_lo, nq_hi;  // -q = nq_hi 2^32 + nq_lo, nq_lo signed
    int32_t M;             // floor(2^(64 + sh) / q)
    uint32_t sh;           // max(0, bits(q) - 47)
    uint32_t prime, off;   // prime index, limb offset in the output
    uint32_t flags, pad;
};

// one conversion of a launch: a ModUp digit, or a ModDown's P limbs
struct MfDigit {
    const MfSlot* slots;
    const uint64_t* tab;         // [n_grp][ks][2][64] 16-byte operands
    uint64_t in_off, out_off;    // words from the batch item's base to the first source limb / the output
    uint32_t n_in, n_out, n_grp;
    uint32_t open;  // bit per group: its primes are all below 2^56 (unreduced butterflies)
};

struct MfArgs {
    MfDigit dig[kMfMaxDigits];
    uint32_t n_dig, n_grp;  // conversions, their groups in all
    uint64_t in_bstride, out_bstride, extra_bstride;
};

hipError_t launch_bconv_ntt_a(const Context& ctx, uint32_t ks, const uint64_t* in, const uint64_t* extra, uint64_t* out,
                              const MfArgs& ma, uint32_t B, const char* name, hipStream_t st);
hipError_t launch_mf_table(const Context& ctx, const uint64_t* cmat, const MfSlot* slots, uint64_t* tab, uint32_t n_in,
                           uint32_t n_out, uint32_t n_grp, uint32_t ks, hipStream_t st);
hipError_t launch_moddown_head(const Context& ctx, const uint64_t* y, uint64_t y_bstride, uint64_t* ehead,
                               uint64_t e_bstride, const uint64_t* xlast, uint64_t x_bstride, const uint64_t* addc,
                               const MfHeadArgs& ha, uint32_t n_polys, hipStream_t st);

}  // namespace fhe
