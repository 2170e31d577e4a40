// swiftkv_exact.hpp -- the integer-compatibility step's arithmetic, shared by
// its two kernels (swiftkv_exact.hip, swiftkv_exact_short.hip): the reference's
// Q15.17 rules (swiftkv_attention.cpp:934-1880;
// llama2_decoder_sw_emulator.cpp:633-711) and the wave scans they use.
#pragma once

#include "swiftkv_device.hpp"

namespace swiftkv {
namespace exact {

using namespace dev;

constexpr int64_t kScoreScaleQ17 = 11585;     // RNE(2^17 / sqrt(128)) (swiftkv_attention.cpp:1101-1102)
constexpr int64_t kLog2eQ21 = 3025551;        // RNE(log2(e) * 2^21) (cpp:207-208)

__device__ __forceinline__ int64_t wrap_bits(int64_t x, int bits) {
    const uint64_t mask = (1ull << bits) - 1u;
    uint64_t r = static_cast<uint64_t>(x) & mask;
    if ((r >> (bits - 1)) & 1u) r |= ~mask;
    return static_cast<int64_t>(r);
}

// Round-half-even of x / 2^s (AP_RND_CONV), 1 <= s <= 31.  With q =
// floor(x / 2^s) and r = x - q 2^s: r < 2^(s-1) gives q, r > 2^(s-1) gives
// q + 1, and the tie gives q + (q & 1) -- all three are floor((x + 2^(s-1) - 1
// + (q & 1)) / 2^s), for either sign of x.  RNE of the exact quotient is odd-
// symmetric, so this equals rounding the magnitude and restoring the sign.
__device__ __forceinline__ int64_t rne_shift(int64_t x, int s) {
    return (x + ((int64_t{1} << (s - 1)) - 1) + ((x >> s) & 1)) >> s;
}

// Q15.17 x unsigned Q1.17 multiplier, RNE >> 17, wrapped to 32 bits.
__device__ __forceinline__ int32_t mulq17_wrap(int32_t a, uint32_t b) {
    return static_cast<int32_t>(static_cast<uint32_t>(
        rne_shift(static_cast<int64_t>(a) * static_cast<int64_t>(b), 17)));   // low 32 bits = the wrap
}

// exp(x) for x <= 0 in Q1.17 through the 33-entry Q30 exp2 table with 12-bit
// linear interpolation (swiftkv_attention.cpp:185-260).  The reference's steps
// with what cannot happen for x <= 0 left out, equal to them for every such x:
//   - l = RNE(x log2(e) 2^-21) in its 24 bits: the product has at most 54
//     significant bits, of which those past the 44 that x > -32.0 needs only
//     decide that the result is 0, so the double product rounds as the integer
//     one wherever that matters, and l > -2^23 there;
//   - below -32.0 the shift is past 31 and the result 0, as the rule has it
//     (both checked against the rule over every x above -40.0);
//   - x = 0 gives l = 0 and 2^17, the shift is at least 13, and the result fits
//     18 bits.
__device__ __forceinline__ uint32_t exp_neg_q17(int32_t x, const uint32_t* lut) {
    int32_t l;   // a saturating conversion
    asm("v_cvt_i32_f64 %0, %1"
        : "=v"(l)
        : "v"(__builtin_rint(static_cast<double>(x) * (static_cast<double>(kLog2eQ21) * 0x1p-21))));
    const uint32_t f = static_cast<uint32_t>(l) & 0x1ffffu;
    const uint32_t idx = f >> 12, rm = f & 0xfffu;
    const uint32_t base = lut[idx], next = lut[idx + 1];
    const uint32_t interp = base + static_cast<uint32_t>((static_cast<uint64_t>(next - base) * rm + (1u << 11)) >> 12);
    const int sh = 13 - (l >> 17);
    return sh < 32 ? (interp + (1u << ((sh - 1) & 31))) >> (sh & 31) : 0u;
}

// 44-bit token dot contribution of one 16-channel half-group, scaled by
// 2^(shift-10) with a floor (cpp:934-995); modulo 2^64, of which the score
// takes 44 bits.
__device__ __forceinline__ int64_t scaled_half(int64_t s, uint32_t shift) {
    return shift >= 10 ? static_cast<int64_t>(static_cast<uint64_t>(s) << ((shift - 10) & 63)) : (s >> (10 - shift));
}

__device__ __forceinline__ int32_t score_of(int64_t token_dot) {
    return sat32(rne_shift(wrap_bits(token_dot, 44) * kScoreScaleQ17, 24));
}

__device__ __forceinline__ uint32_t shift_of(float scale) { return (__float_as_uint(scale) >> 23) - 110u; }

// The single-pass recurrence (cpp:1276-1335, 1463-1558).  Word of a token:
constexpr uint32_t kInit = 1u << 31;      // first token of the sequence: Y = v, Z = 1
constexpr uint32_t kRescale = 1u << 30;   // new maximum: Y = Y * coef + v, Z = Z * coef + 1
constexpr uint32_t kCoefMask = (1u << 18) - 1u;
constexpr uint32_t kMask30 = (1u << 30) - 1u;

// Coefficient word of a token with score s and prefix maximum `before`.
__device__ __forceinline__ uint32_t coef_word(int32_t s, int32_t before, const uint32_t* lut) {
    const int32_t x = __builtin_elementwise_sub_sat(min(s, before), max(s, before));
    return exp_neg_q17(x, lut) | (s > before ? kRescale : 0u);
}

// Z in Q13.17, wrapped to 30 bits.
__device__ __forceinline__ uint32_t z_step(uint32_t z, uint32_t word) {
    if (word & kInit) return 1u << 17;
    const uint32_t coef = word & kCoefMask;
    if (word & kRescale)
        return ((static_cast<uint32_t>(rne_shift(static_cast<int64_t>(z) * coef, 17)) & kMask30) + (1u << 17)) &
               kMask30;
    return (z + coef) & kMask30;
}

// Y per token and channel (cpp:1463-1558), v = code << shift as the
// reference's ap_int<32> (it wraps for code 64, shift 25):
//   first token  Y = v
//   no rescale   Y = sat32(Y + wrap32(RNE(v c >> 17)))
//   rescale      Y = sat32(wrap32(RNE(Y c >> 17)) + v)
__device__ __forceinline__ int32_t dequant_raw(int32_t code, uint32_t shift) {
    return static_cast<int32_t>(static_cast<uint32_t>(code) << (shift & 31u));
}
__device__ __forceinline__ int32_t y_step(int32_t y, uint32_t word, int32_t v) {
    if (word & kInit) return v;
    const uint32_t coef = word & kCoefMask;
    if (word & kRescale) return __builtin_elementwise_add_sat(mulq17_wrap(y, coef), v);
    return __builtin_elementwise_add_sat(y, mulq17_wrap(v, coef));
}

// The term of an ordinary token as one fused multiply-add: with p = c 2^(s-17),
// the product of the coefficient c (at most 2^17) and the V scale (exact in
// FP32), it is RNE(code p).  For a shift of at most 15 (V groups below 32.0,
// the common case) |code p| <= 128 2^15 = 2^22, so code p + 1.5 2^23 lies in
// [2^23, 2^24), where the floats are the integers: the addition rounds the
// exact sum once, to nearest even, and 1.5 2^23 is an even integer, so the
// result's bits are 0x4b400000 + RNE(code p).  Larger shifts take the 64-bit
// integer form.
constexpr float kRoundMagic = 12582912.0f;   // 1.5 * 2^23
constexpr uint32_t kRoundMagicBits = 0x4b400000u;
constexpr float kWideScale = 0.5f;           // V scale of shift 16
constexpr float kHugeScale = 128.0f;         // V scale of shift 24
__device__ __forceinline__ uint32_t term_bits(int32_t code, float p) {
    return __float_as_uint(__builtin_fmaf(static_cast<float>(code), p, kRoundMagic));
}

// Sum over the 8 lanes of an aligned octet of a 64-bit integer (DPP moves of
// both halves, integer adds, so exact in any order); every lane gets it.
template <int Ctrl>
__device__ __forceinline__ int64_t dpp64(int64_t x) {
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), Ctrl, 0xF, 0xF, true));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x >> 32), Ctrl, 0xF, 0xF, true));
    return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}
__device__ __forceinline__ int64_t octet_sum64(int64_t x) {
    x += dpp64<kDppQuadXor1>(x);
    x += dpp64<kDppQuadXor2>(x);
    return x + dpp64<kDppHalfMirror>(x);
}

// Inclusive wave scans with DPP (GFX9): row shifts by 1, 2, 4, 8 scan each
// 16-lane row, then row 0's last lane is broadcast into row 1 and row 2's
// into row 3, then lane 31 into rows 2 and 3.  Lanes a move cannot reach, and
// rows outside its row mask, take the identity.
constexpr int kDppRowShr1 = 0x111, kDppRowShr2 = 0x112, kDppRowShr4 = 0x114, kDppRowShr8 = 0x118;
constexpr int kDppRowBcast15 = 0x142, kDppRowBcast31 = 0x143, kDppWaveShr1 = 0x138;

template <int Ctrl, int RowMask>
__device__ __forceinline__ int32_t dpp_shifted(int32_t identity, int32_t x) {
    return __builtin_amdgcn_update_dpp(identity, x, Ctrl, RowMask, 0xF, false);
}

__device__ __forceinline__ int32_t wave_scan_max(int32_t x) {
    x = max(x, dpp_shifted<kDppRowShr1, 0xF>(INT32_MIN, x));
    x = max(x, dpp_shifted<kDppRowShr2, 0xF>(INT32_MIN, x));
    x = max(x, dpp_shifted<kDppRowShr4, 0xF>(INT32_MIN, x));
    x = max(x, dpp_shifted<kDppRowShr8, 0xF>(INT32_MIN, x));
    x = max(x, dpp_shifted<kDppRowBcast15, 0xA>(INT32_MIN, x));
    return max(x, dpp_shifted<kDppRowBcast31, 0xC>(INT32_MIN, x));
}

__device__ __forceinline__ uint32_t wave_scan_add(uint32_t v) {
    int32_t x = static_cast<int32_t>(v);
    x += dpp_shifted<kDppRowShr1, 0xF>(0, x);
    x += dpp_shifted<kDppRowShr2, 0xF>(0, x);
    x += dpp_shifted<kDppRowShr4, 0xF>(0, x);
    x += dpp_shifted<kDppRowShr8, 0xF>(0, x);
    x += dpp_shifted<kDppRowBcast15, 0xA>(0, x);
    return static_cast<uint32_t>(x + dpp_shifted<kDppRowBcast31, 0xC>(0, x));
}

__device__ __forceinline__ float wave_scan_add(float v) {
    auto from = [](float x, auto move) { return __int_as_float(move(__float_as_int(x))); };
    v += from(v, [](int32_t x) { return dpp_shifted<kDppRowShr1, 0xF>(0, x); });
    v += from(v, [](int32_t x) { return dpp_shifted<kDppRowShr2, 0xF>(0, x); });
    v += from(v, [](int32_t x) { return dpp_shifted<kDppRowShr4, 0xF>(0, x); });
    v += from(v, [](int32_t x) { return dpp_shifted<kDppRowShr8, 0xF>(0, x); });
    v += from(v, [](int32_t x) { return dpp_shifted<kDppRowBcast15, 0xA>(0, x); });
    return v + from(v, [](int32_t x) { return dpp_shifted<kDppRowBcast31, 0xC>(0, x); });
}

}  // namespace exact
}  // namespace swiftkv
