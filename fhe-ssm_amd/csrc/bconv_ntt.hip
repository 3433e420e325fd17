// bconv_ntt.hip -- the approximate CRT basis conversion (BConv) of ModUp and ModDown on the matrix cores, fused with
// the first pass of the forward NTT that reads its outputs.
//
// out_j[k] = sum_i y_i[k] c_ij mod p_j is a contraction over the source limbs i whose constants are shared by all
// 65,536 coefficients, so it runs as int8 MFMAs: y_i is split into 8 balanced base-256 digits y_i = sum_p 256^p d_ip
// (d_ip in [-128, 127], so the word (y + 0x80..80) ^ 0x80..80 holds them as signed bytes), and 256^p moves into the
// constants, C_ijp = 256^p c_ij mod p_j, themselves split into 8 balanced digits.  Then
//     V_j = sum_{i,p} d_ip C_ijp = sum_s 256^s D_js,   D_js = sum_{i,p} d_ip (digit s of C_ijp),
// is congruent to the wanted sum, and the eight D_js of an output are rows of one integer matrix product over the
// 8 n_in bytes of the inputs: one 16x16x64 MFMA takes 8 source limbs, 16 coefficients and 16 of the 8 n_out rows.  Rows
// are dealt so that lane (g, n) (g = lane / 16) of a pair of MFMAs ends up with all eight D of output 4 grp + g at
// coefficient n; |V| < 2^10 n_in p_j, and one quotient estimate brings it to [0, 2 p_j) (mf_reduce): 14 VALU instructions
// an output word, where three 64-bit multiply-adds a term and a Montgomery reduction took 58.  A ModDown adds a signed
// integer of its own to the sum (the rounding correction and the rescale's lifted limb, k_moddown_head).
//
// The source words arrive as digit words: the inverse NTT that produces them multiplies by qhat_i^-1 along with N^-1 in
// its last stage (JobSpec.scale) and stores the digits, so no word is converted more than once.
//
// A wave forms 4 outputs of one column (the 256 words c + 256 r) straight into the registers of the NTT's first pass
// (lane (g, n): output g, rows n + 16 k), runs its 8 stages (radix 16, an exchange between the 16 lanes of an output
// through the wave's own LDS, radix 16) and stores the intermediate the second pass reads: the converted limbs never make
// a round trip through memory of their own, and no barrier joins the waves.  Sources and outputs are column-major within 16
// rows, the second pass's tiles (word c + 256 r at 4096 (r / 16) + 16 c + r % 16), so that every access is of 128
// consecutive bytes: with row-major limbs and workgroup tiles of 8 columns, whose 64-byte pieces of lines cost full ones,
// the same conversion took 1,515 us.
//
// Measured (64 x 3 digits, 8 -> 24 limbs of 54 and 60 bits): 1,093-1,178 us, where the conversion on the VALU (739 us,
// VALU-bound) and the separate first pass (974 us) took 1,713; 128 ModDowns of 8 -> 23 limbs 811-882 us and their head
// 146-152, before 569 and 669.  What bounds it: 451 M VALU wave instructions (71 of the 96 an output word are the
// butterflies), 0.96 ms at the issue rate of the 1.84 GHz that it holds, over 3.2 GB of memory traffic.  With few outputs
// the VALU form is the faster one: the rule and its measurements are at mf_modup and mf_moddown in ops.cpp.
#include <algorithm>

#include "bconv_ntt.hpp"
#include "engine.hpp"
#include "ks_device.hpp"
#include "modarith.hpp"
#include "ntt_device.hpp"

namespace fhe {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr uint64_t kDigitBias = 0x8080808080808080ull;
constexpr int kBcWaves = 4;         // waves of a workgroup: adjacent columns
constexpr int kBcLds = 4 * 272;     // LDS words of a wave: 4 outputs x 256 rows, one word of padding per 16

// V = sum_s 256^s D_s (D0: s = 0..3, D1: s = 4..7) + e -> V mod q, in [0, 2q).  |V - e| < 2^14 q (16 inputs), |e| < 2^60.
// With W = floor(V / 2^32) exactly, G = floor(W / 2^sh) and M = floor(2^(64+sh) / q) (sh as in mf_add: |G| < 2^29.6,
// M < 2^31), G M / 2^32 lies in [V/q - 0.44, V/q + 0.19]; its floor after subtracting a quarter is a quotient k with
// V - k q in (0, 1.7 q).  V and -k q need their low 64 bits only.
template <bool kExtra>
__device__ __forceinline__ uint64_t mf_reduce(const v4i& D0, const v4i& D1, uint64_t e, const MfSlot& c) {
    const int32_t E0 = D0[0] + (D0[1] << 8), E1 = D0[2] + (D0[3] << 8);
    const int32_t E2 = D1[0] + (D1[1] << 8), E3 = D1[2] + (D1[3] << 8);
    int64_t F = (int64_t)E1 * 65536 + E0;
    if (kExtra) F += (uint32_t)e;
    const int64_t W = (int64_t)E3 * 65536 + ((int32_t)(F >> 32) + E2 + (kExtra ? (int32_t)(e >> 32) : 0));
    const int32_t G = (int32_t)__builtin_amdgcn_alignbit((uint32_t)((uint64_t)W >> 32), (uint32_t)W, c.sh);
    const int32_t k = (int32_t)(((int64_t)G * c.M - (1ll << 30)) >> 32);
    const uint64_t v = ((uint64_t)(uint32_t)W << 32) | (uint32_t)F;
    const uint64_t r = v + (uint64_t)((int64_t)k * c.nq_lo);
    return r + ((uint64_t)((uint32_t)k * (uint32_t)c.nq_hi) << 32);
}

// a word at a byte offset from a wave-uniform base (the load and store forms with a scalar base and a 32-bit offset)
__device__ __forceinline__ uint64_t ld_off(const uint64_t* base, uint32_t byte_off) {
    return *reinterpret_cast<const uint64_t*>(reinterpret_cast<const char*>(base) + byte_off);
}
__device__ __forceinline__ void st_off(uint64_t* base, uint32_t byte_off, uint64_t v) {
    __builtin_nontemporal_store(v, reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(base) + byte_off));
}

// The conversion of one lane's 16 words (rows n + 16 k of output 4 grp + g), KS steps of 8 source limbs.  off[s][h]: byte
// offset of source word (step s, input 2 g + h) of row n from the wave-uniform base.  kTail: the last step has one input
// (h = 1 is not read).  kExtra: the words at ebase + eoff are added.  tv: the lane's twiddle (entry tw of the output's
// prime), requested with the source words.
template <int KS, bool kTail, bool kExtra>
__device__ __forceinline__ void mf_words(uint64_t* x, const uint64_t* base, const uint32_t (&off)[KS][2],
                                         const uint64_t* ebase, uint32_t eoff, const v4i* __restrict__ A, const MfSlot& c,
                                         TwPair& tv, const TwPair* __restrict__ tw) {
    v4i a[KS][2];
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
        for (int t = 0; t < 2; t++) a[s][t] = A[(s * 2 + t) * 64];
    constexpr int kB = KS == 2 || kExtra ? 8 : 16;  // rows whose words are requested together (as registers allow)
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += kB) {
        uint64_t y[kB][KS][2], e[kB];
#pragma unroll
        for (int k = 0; k < kB; k++) {
#pragma unroll
            for (int s = 0; s < KS; s++)
#pragma unroll
                for (int h = 0; h < 2; h++)
                    y[k][s][h] = kTail && s == KS - 1 && h ? 0 : ld_off(base + 4096 * (k0 + k), off[s][h]);
            e[k] = kExtra ? ld_off(ebase + 4096 * (k0 + k), eoff) : 0;
        }
        if (k0 == 0) tv = tw[256 * c.prime];
        __builtin_amdgcn_sched_barrier(0);  // all of them in flight before the first product waits
#pragma unroll
        for (int k = 0; k < kB; k++) {
            v4i D0 = {0, 0, 0, 0}, D1 = {0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const v4i b = {(int)(uint32_t)y[k][s][0], (int)(uint32_t)(y[k][s][0] >> 32),
                               (int)(uint32_t)y[k][s][1], (int)(uint32_t)(y[k][s][1] >> 32)};
                D0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[s][0], b, D0, 0, 0, 0);
                D1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[s][1], b, D1, 0, 0, 0);
            }
            x[k0 + k] = mf_reduce<kExtra>(D0, D1, e[k], c);
        }
    }
}

// the forward NTT's stages 0..3 on rows n + 16 k
template <bool kOpen>
__device__ __forceinline__ void stages03(uint64_t* x, const TwPair* tw, uint64_t q) {
    const uint64_t q4 = q << 2, nq = 0 - q;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int h = 8 >> s;
#pragma unroll
        for (int k = 0; k < 16; k++) {
            if (k & h) continue;
            fwd_bfly<kOpen>(x[k], x[k + h], tw[(1 << s) + (k >> (4 - s))], q4, nq);
        }
    }
}

// stages s0..s1-1 of 4..7 on rows 16 n + k; tw: the stages' 15 pairs, stage s's first at 2^(s-4) - 1
template <bool kOpen>
__device__ __forceinline__ void stages47(uint64_t* x, const TwPair* tw, uint64_t q, int s0, int s1) {
    const uint64_t q4 = q << 2, nq = 0 - q;
#pragma unroll
    for (int s = s0; s < s1; s++) {
        const int h = 128 >> s;
#pragma unroll
        for (int k = 0; k < 16; k++) {
            if (k & h) continue;
            fwd_bfly<kOpen>(x[k], x[k + h], tw[(1 << (s - 4)) - 1 + (k >> (8 - s))], q4, nq);
        }
    }
}

// what a lane wrote to its wave's LDS before is seen by the wave's other lanes after (a wave's LDS operations complete in
// order; the fence keeps the compiler's)
__device__ __forceinline__ void wave_exchange() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

struct BcShared {
    uint64_t x[kBcLds];
    TwPair tw[64];  // stages 0..3's twiddles of the four primes: [output][16]
};

// a wave's part: the four outputs of a group over one column; in, out: the batch item's first source limb and output,
// extra: its added limb
template <int KS, bool kTail, bool kExtra, bool kOpen>
__device__ __forceinline__ void bc_column(const uint64_t* __restrict__ in, const uint64_t* __restrict__ extra,
                                          uint64_t* __restrict__ out, const MfSlot* __restrict__ slots,
                                          const v4i* __restrict__ tab, uint32_t n_in, uint32_t col, BcShared& sh,
                                          const TwPair* __restrict__ twa) {
    // (opaque per instance: otherwise the addresses that the open and the other instance share are formed before their
    // branch and kept, spilled, through one for the other)
    uint32_t lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const uint32_t g = lane >> 4, n = lane & 15;
    uint64_t x[16];
    const uint32_t w = 16 * col + n;
    uint32_t off[KS][2];
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            // inputs past the last have zero constants: any readable word will do (the last one's: the same lines)
            const uint32_t i = min(s * 8 + 2 * g + h, n_in - 1);
            off[s][h] = (i * kN + w) * 8;
        }
    const MfSlot c = slots[g];
    TwPair tv;
    mf_words<KS, kTail, kExtra>(x, in, off, extra, w * 8, tab + lane, c, tv, twa + n);
    sh.tw[lane] = tv;
    wave_exchange();
    stages03<kOpen>(x, sh.tw + 16 * g, c.q);
    // rows 16 n + k: the twiddles of stages 4..6 are requested before the exchange, stage 7's after it.  Stage s's entry
    // 2^s + 2^(s-4) n + j of the plain table stands at 2^s + 16 j + n of this kernel's (twa), so that a load's 16 lanes of
    // an output read 256 consecutive bytes (in the plain table stage 7's lanes are a line apart, and the loads took a fifth
    // of the kernel's time)
    const TwPair* tw = twa + 256 * c.prime + n;
    TwPair tw47[15];
#pragma unroll
    for (int s = 4, m = 0; s < 7; s++)
#pragma unroll
        for (int j = 0; j < (1 << (s - 4)); j++, m++) tw47[m] = tw[(1 << s) + 16 * j];
    uint64_t* L = sh.x + 272 * g;
#pragma unroll
    for (int k = 0; k < 16; k++) L[n + 17 * k] = x[k];
    wave_exchange();
#pragma unroll
    for (int j = 0; j < 8; j++) tw47[7 + j] = tw[128 + 16 * j];
#pragma unroll
    for (int k = 0; k < 16; k++) x[k] = L[17 * n + k];
    wave_exchange();
    stages47<kOpen>(x, tw47, c.q, 4, 8);
    // back to rows n + 16 k: stores of 128 consecutive bytes an output
#pragma unroll
    for (int k = 0; k < 16; k++) L[17 * n + k] = x[k];
    wave_exchange();
    if (c.flags & kMfNone) return;  // a group's unused slot
    const uint32_t bo = (c.off * kN + w) * 8;  // an item's output spans less than 4 GiB
#pragma unroll
    for (int k = 0; k < 16; k++) st_off(out + 4096 * k, bo, L[n + 17 * k]);
}

// grid: 64 quads of columns x (groups of 4 outputs of every digit) x batch, one dimension.  Workgroups go to the 8 XCDs
// round-robin; id = xcd + 8 s, and XCD xcd takes the columns [32 xcd, 32 xcd + 32), s running over their 8 quads fastest,
// then the groups (which read the same source words, kept by that XCD's L2), then the batch.
// Two steps of source limbs run three waves a SIMD with 8 rows' words in flight: 140 to 156 registers, and 168 with 3
// spilled for 10 to 16 limbs with an added one; four waves with 4 rows' have 128 and spill 3 to 10.  Three against four, us
// (whole levels of 54- and 60-bit chains, 16 x 2 digits or 32 ModDowns): 16 limbs 337 / 361 ModUp, 314 / 319 ModDown, 311-324
// / 346 exact; 12 limbs 256 / 272, 234 / 236, 226-237 / 253; 9 limbs 197-202 / 202, 179 / 179, 168 / 162.
template <int KS, bool kTail, bool kExtra>
__global__ __launch_bounds__(64 * kBcWaves) __attribute__((amdgpu_waves_per_eu(KS == 2 ? 3 : 4))) void k_bconv_ntt_a(
    const uint64_t* __restrict__ in, const uint64_t* __restrict__ extra, uint64_t* __restrict__ out, MfArgs ma,
    const TwPair* __restrict__ twa) {
    __shared__ BcShared shared[kBcWaves];
    const uint32_t id = blockIdx.x, s0 = id >> 3, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t col = ((id & 7) * 8 + (s0 & 7)) * kBcWaves + wave, gi = s0 >> 3;
    const uint32_t b = uni_div(gi, ma.n_grp);
    uint32_t grp = gi - b * ma.n_grp, d = 0;
    while (d + 1 < ma.n_dig && grp >= ma.dig[d].n_grp) grp -= ma.dig[d++].n_grp;
    const MfDigit& dg = ma.dig[d];
    const MfSlot* slots = dg.slots + 4 * grp;
    const uint64_t* src = in + b * ma.in_bstride + dg.in_off;
    const uint64_t* ex = kExtra ? extra + b * ma.extra_bstride : nullptr;
    uint64_t* dst = out + b * ma.out_bstride + dg.out_off;
    const v4i* tab = reinterpret_cast<const v4i*>(dg.tab) + (size_t)grp * (KS * 2 * 64);
    BcShared& sh = shared[wave];
    if (dg.open >> grp & 1)  // all four primes take the open butterflies
        bc_column<KS, kTail, kExtra, true>(src, ex, dst, slots, tab, dg.n_in, col, sh, twa);
    else
        bc_column<KS, kTail, kExtra, false>(src, ex, dst, slots, tab, dg.n_in, col, sh, twa);
}

// the MFMA operand table of a plan from its constants: cmat [n_in][n_out] (c_ij mod p_j, plain residues).  Lane
// (kb = lane / 16, m = lane % 16) of MFMA t holds row m -- digit s = 4 t + m % 4 of output 4 grp + m / 4 -- over the bytes
// of inputs 2 kb, 2 kb + 1 of a step.  One thread per (group, step, t, lane).
__global__ __launch_bounds__(256) void k_mf_table(const uint64_t* __restrict__ cmat, const MfSlot* __restrict__ slots,
                                                  uint64_t* __restrict__ tab, uint32_t n_in, uint32_t n_out, uint32_t ks,
                                                  uint32_t n_thr, const PrimeInfo* __restrict__ primes) {
    const uint32_t id = blockIdx.x * 256 + threadIdx.x;
    if (id >= n_thr) return;
    const uint32_t lane = id & 63, t = (id >> 6) & 1, st = id >> 7, step = st % ks, grp = st / ks;
    const uint32_t m = lane & 15, o = grp * 4 + (m >> 2), s = 4 * t + (m & 3);
    for (uint32_t h = 0; h < 2; h++) {
        const uint32_t i = step * 8 + 2 * (lane >> 4) + h;
        uint64_t w = 0;
        if (i < n_in && o < n_out) {
            const Barrett br = barrett_of(primes[slots[o].prime]);
            uint64_t C = cmat[(size_t)i * n_out + o];
            for (uint32_t p = 0; p < 8; p++) {
                const uint64_t dg = (C + kDigitBias) ^ kDigitBias;
                w |= ((dg >> (8 * s)) & 0xFFull) << (8 * p);
                C = reduce128(C >> 56, C << 8, br);  // C < 2^60: C >> 56 < 16 < q
            }
        }
        tab[(size_t)id * 2 + h] = w;
    }
}

// The part of a ModDown that needs all P limbs of a coefficient at once: the exact form's rounding correction
// u = round(sum_i y_i / p_i), and with a rescale the dropped limb's value z = addc + (x_{l-1} - conv_{l-1}) P^-1 mod
// q_{l-1}, lifted to z' in (-q/2, q/2].  Both enter the conversion, whose columns carry P^-1, as one signed integer
// e = z' - u (z' or -u alone when only one applies), |e| < 2^59 + 16.  y: the P limbs as digit words.
__global__ __launch_bounds__(256) void k_moddown_head(const uint64_t* __restrict__ y, uint64_t y_bstride, uint64_t* ehead,
                                                      uint64_t e_bstride, const uint64_t* xlast, uint64_t x_bstride,
                                                      const uint64_t* __restrict__ addc, MfHeadArgs ha,
                                                      const PrimeInfo* __restrict__ primes) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x, b = blockIdx.y;
    const uint64_t* src = y + b * y_bstride + k;
    uint64_t yv[kMfMaxIn];
#pragma unroll
    for (int i = 0; i < kMfMaxIn; i++)
        if (i < (int)ha.n_in) yv[i] = (src[(size_t)i * kN] ^ kDigitBias) - kDigitBias;
    uint64_t u = 0;
    if (ha.exact) {
        U128 F{0, 0};  // sum of floor(y_i floor(2^128 / p_i) / 2^64)
#pragma unroll
        for (int i = 0; i < kMfMaxIn; i++)
            if (i < (int)ha.n_in) {
                mac128(F, yv[i], ha.fix[i][1]);
                const uint64_t h = mulhi64(yv[i], ha.fix[i][0]);
                F.lo += h;
                F.hi += (F.lo < h) ? 1 : 0;
            }
        const uint64_t lo = F.lo + (1ull << 63);
        u = F.hi + (lo < F.lo ? 1 : 0);
    }
    uint64_t e = 0 - u;
    if (ha.rescale) {
        const Barrett bl = barrett_of(primes[ha.last]);
        const uint64_t ql = bl.q;
        Acc s;
#pragma unroll
        for (int i = 0; i < kMfMaxIn; i++)
            if (i < (int)ha.n_in) {
                s.add(yv[i], ha.c[i]);
                if (i == 7) s.fold();
            }
        s.fold();
        s.add(u, ha.c[kMfMaxIn]);  // - u P: the constant is -P mod q_{l-1}
        const uint64_t conv = reduce_u128(s.get(), bl);
        uint64_t z = shoup(sub_mod(xlast[b * x_bstride + k], conv, ql), ha.pinv.w, ha.pinv.wp, ql);
        if (addc) z = add_mod(z, addc[(size_t)b * kN + k], ql);
        e += z - (z > (ql >> 1) ? ql : 0);
    }
    ehead[b * e_bstride + k] = e;
}

}  // namespace

hipError_t launch_bconv_ntt_a(const Context& ctx, uint32_t ks, const uint64_t* in, const uint64_t* extra, uint64_t* out,
                              const MfArgs& ma, uint32_t B, const char* name, hipStream_t st) {
    if (B == 0) return hipSuccess;
    if (ks < 1 || ks > 2 || ma.n_dig == 0 || ma.n_dig > kMfMaxDigits || ma.n_grp == 0) return hipErrorInvalidValue;
    // algorithmic bytes: inputs read once, outputs written
    double limbs = 0;
    bool tail = true;
    for (uint32_t d = 0; d < ma.n_dig; d++) {
        if (ma.dig[d].n_in == 0 || ma.dig[d].n_in > 8 * ks) return hipErrorInvalidValue;
        tail = tail && ma.dig[d].n_in <= 9;
        limbs += ma.dig[d].n_in + ma.dig[d].n_out + (extra ? 1 : 0);
    }
    const int pi = prof_begin(ctx, name, limbs * B * kN * 8, st);
    const dim3 grid(256 / kBcWaves * ma.n_grp * B), block(64 * kBcWaves);
    auto k = ks == 1 ? (extra ? k_bconv_ntt_a<1, false, true> : k_bconv_ntt_a<1, false, false>)
             : tail  ? (extra ? k_bconv_ntt_a<2, true, true> : k_bconv_ntt_a<2, true, false>)
                     : (extra ? k_bconv_ntt_a<2, false, true> : k_bconv_ntt_a<2, false, false>);
    hipLaunchKernelGGL(k, grid, block, 0, st, in, extra, out, ma, ctx.d_twa);
    prof_end(ctx, pi, st);
    return hipGetLastError();
}

hipError_t launch_mf_table(const Context& ctx, const uint64_t* cmat, const MfSlot* slots, uint64_t* tab, uint32_t n_in,
                           uint32_t n_out, uint32_t n_grp, uint32_t ks, hipStream_t st) {
    const uint32_t n_thr = n_grp * ks * 128;
    hipLaunchKernelGGL(k_mf_table, dim3((n_thr + 255) / 256), dim3(256), 0, st, cmat, slots, tab, n_in, n_out, ks, n_thr,
                       ctx.d_primes);
    return hipGetLastError();
}

hipError_t launch_moddown_head(const Context& ctx, const uint64_t* y, uint64_t y_bstride, uint64_t* ehead,
                               uint64_t e_bstride, const uint64_t* xlast, uint64_t x_bstride, const uint64_t* addc,
                               const MfHeadArgs& ha, uint32_t n_polys, hipStream_t st) {
    if (ha.n_in == 0 || ha.n_in > (uint32_t)kMfMaxIn || (ha.rescale && !xlast)) return hipErrorInvalidValue;
    const double limbs = ha.n_in + 1 + (ha.rescale ? 1 : 0) + (addc ? 1 : 0);
    const int pi = prof_begin(ctx, "bconv_head", limbs * n_polys * kN * 8, st);
    hipLaunchKernelGGL(k_moddown_head, dim3(kN / 256, n_polys), dim3(256), 0, st, y, y_bstride, ehead, e_bstride, xlast,
                       x_bstride, addc, ha, ctx.d_primes);
    prof_end(ctx, pi, st);
    return hipGetLastError();
}

}  // namespace fhe
