// swiftkv_exact.hip -- integer-compatibility step: the reference's Q15.17
// single-pass recurrence evaluated exactly on the GPU, so the A14 words and
// E8M0 codes equal the reference's bit for bit (swiftkv_attention.cpp:934-1880;
// llama2_decoder_sw_emulator.cpp:633-711).
//
// The recurrence over (max, Z, Y) looks sequential, but only the tokens that
// raise the running maximum (about ln n of n) must be taken in order:
//   - the running maximum before a token is the prefix maximum of the scores,
//     so all scores come first, then every coefficient at once;
//   - an ordinary token adds a term to Y and its coefficient to Z that depend
//     on neither; while no partial sum of Y can reach an end of the int32 range
//     the saturating adds are plain adds, and a sum modulo 2^32 in any order is
//     the reference's.  Each sum carries a bound of its terms' magnitudes; where
//     |Y| plus the bound could reach 2^31 the range goes through the ordered pass.
//
// One 8-wave workgroup per CU.  Launches that split heads have the grid
// (splits, 32 heads, batch rows); workgroup (j, h, z) owns tokens [j*C,
// min((j+1)*C, position)) of head h of rows[z]'s sequence.  The others have up
// to one workgroup per CU, each taking whole heads in turn.  Per head:
//   1. every wave loads its first K and V blocks (64 tokens: lane = chunk c =
//      lane&7 of 16 channels, row r = lane>>3 of 8 rows), then rotates the
//      query and splits it into signed-byte limbs; the last wave also quantizes
//      the new row and scores it (the owner of `position` appends it);
//   2. K pass: scores of the wave's blocks (round-robin) into LDS, with each
//      block's maximum and the V scales' exponents;
//   3. the block maxima are exchanged (LDS barrier; with several splits, one
//      tagged word per split): the running maximum before every block, and which
//      blocks hold a new one ("hot": usually three or four beyond the first);
//   4. V pass: coefficients of the wave's blocks, then V codes straight from
//      memory times coefficient times scale, rounded per term, summed per lane.
//      A wave's sums go to LDS where a stretch between hot blocks ends; of a hot
//      block, the tokens from its first to its last new maximum are left to 5,
//      as terms in LDS;
//   5. Y is folded over those few sums and terms in token order by one thread
//      per channel, Z by one wave; the new token is the last step, then Y * 1/Z
//      and the integer-path A14/E8M0 epilogue.
// The next head's first blocks are loaded behind the last ones of this head, so
// that the fold and the prologue run under them.
//
// With several splits, each publishes its sums and new maxima as tagged words,
// and the last of a head to arrive folds them (the fast step's exchange).  A
// split that cannot publish in full -- it did not hear of the maxima before it
// in time, or has too many new ones -- says so, and then, or where a bound
// fails, the last to arrive runs the head from that split on by itself: no wait
// is unbounded and no result depends on who waits for whom.
//
// The ordered pass takes what the sums cannot carry, token by token: hot blocks
// past the staging rows, ranges where a sum could saturate Y, splits with too
// many new maxima.  Heads of rising scores (recency, drift) depend on it, so all
// eight waves work at it: five stage terms in LDS while three run Y and Z over
// the round before.
//
// What bounds it: for small batches the chain of round trips (first loads, K
// pass, exchange of maxima, V pass, fold, exchange of sums); for large ones the
// stream, at 6.9 TB/s within the K and V passes of a head, with about 7 us of
// fold, barriers and ramps per 50 us head.  Calls back to back on one set of
// buffers, context 4096, N(0, 1), us per call, the chunked kernel it replaced (Y
// in token order through LDS, up to four workgroups per head each scoring every
// token) against this one:
//   batch     1            2            4            8            16           32           64
//   normal    90.6 / 23.8  93.4 / 26.7  87.5 / 36.9  113 / 55.3   135 / 104    233 / 197    433 / 380
//   scores that rise by 8 sigma over the last 200 tokens:
//             103 / 35.0   108 / 45.4   100 / 69.5   123 / 59.9   146 / 112    241 / 215    446 / 413
//   every token a new maximum:
//             557 / 115    557 / 119    517 / 128    542 / 140    582 / 271    632 / 535    1243 / 1042
// Slower than that kernel, which took every token from LDS at one rate: Y that
// saturates for thousands of tokens, from batch 16 on (141 / 188, at 64 439 / 709),
// and scores that drift by 16 sigma and more over the context, from batch 32 on
// (462 / 483 at 64; 272 / 318 at 64 and context 2048).
// Tried: two 8-wave workgroups per CU (128 registers, 480 at batch 64: their
// streams get in each other's way, and a batch-1 launch then doubles workgroups
// up on half the CUs, 39 against 28);
// reloading each row as soon as it is used (426 against 431, but the compiler
// gives the rows other registers in each loop and waits for all loads to copy
// them); sums per piece between new maxima (a masked pass and a reduction each,
// 5-6 us per head more).
#include <algorithm>
#include <type_traits>

#include "swiftkv_exact.hpp"

namespace swiftkv {
namespace {

using namespace exact;

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kBlock = 64;                    // tokens a wave takes at a time
constexpr int kRows = kBlock / 8;             // token rows per lane of a block
constexpr int kMaxBlocks = kExactMaxTokens / kBlock;
static_assert(kMaxBlocks <= 64, "one lane per block where the block maxima are scanned");
// Accumulators per workgroup: one per stretch between hot blocks and cuts (up
// to 65), and in a split that cannot fold its own sums one per special token,
// from the back.  4096 tokens in random order hold 8.9 +- 2.8 new maxima in
// about five hot blocks.
constexpr int kPool = 65 + kExactEntries - 1;
constexpr int kSpecials = kExactEntries - 1;
constexpr int kStageRows = 128;               // tokens of hot blocks staged in LDS

// 16 rotated query channels as signed-byte limbs, q = l0 + l1 2^8 + l2 2^16 +
// l3 2^24 + l4 2^32 (each limb in [-128, 127]): a lane holds limbs 0-2 of its
// chunk's channels, four to a word; limbs 3 and 4 stay in LDS, as they are zero
// for |q| below about 64.0.
struct QueryLimbs {
    int32_t w[3][4];
};

// Exact dot of 16 codes with limbs 0-2 of the query (|sum| < 2^35).
__device__ __forceinline__ double limb_dot3(const QueryLimbs& L, v4i k) {
    int32_t s[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        int32_t acc = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_sdot4(L.w[i][j], k[j], acc, false);
        s[i] = acc;
    }
    return __builtin_fma(static_cast<double>(s[2]), 65536.0, static_cast<double>(s[0] + s[1] * 256));
}

__device__ __forceinline__ double octet_sum_f64(double x) {
    x += __builtin_bit_cast(double, dpp64<kDppQuadXor1>(__builtin_bit_cast(int64_t, x)));
    x += __builtin_bit_cast(double, dpp64<kDppQuadXor2>(__builtin_bit_cast(int64_t, x)));
    return x + __builtin_bit_cast(double, dpp64<kDppHalfMirror>(__builtin_bit_cast(int64_t, x)));
}

// Orders a wave's LDS writes before its own later reads of what other lanes
// wrote (the hardware runs a wave's LDS operations in order).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A wave-uniform value the compiler cannot see is uniform (it came through LDS
// or memory), moved to a scalar register: control flow and buffer offsets that
// depend on it stay scalar.
__device__ __forceinline__ int32_t uniform(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint32_t uniform(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}

__device__ __forceinline__ int8_t* uniform(int8_t* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    return reinterpret_cast<int8_t*>(static_cast<uint64_t>(uniform(static_cast<uint32_t>(v >> 32))) << 32 |
                                     uniform(static_cast<uint32_t>(v)));
}

// ---------------------------------------------------------------- state

struct Shared {
    // Per token of the range: x is the score, then the coefficient as a float
    // (sign set for a first or rescaling token, zero past the range); y the
    // biased exponents of the token's four V scales, a byte each.
    uint2 tok[kExactMaxTokens + 2];               // and one that adds nothing, for the ordered pass
    // Sums of ordinary terms, modulo 2^32, of the coefficients, and of
    // coefficient times scale per group (the bound).
    int32_t pool[kPool][kHeadDim];
    uint32_t pool_z[kPool];
    __attribute__((aligned(16))) float pool_b[kPool][kGroupsPerHead];
    // Folding workgroups, per hot block: its tokens from the first to the last
    // special one, {first token | past the last << 16, row of `stage` where
    // they start (not staged if they would end past it), what Y is multiplied
    // by at the first}; per staged token what Y is multiplied by (Q1.17, 1.0 for
    // an ordinary one; a float in the ordered pass) and what is added to it and
    // to Z.
    uint4 hot[kPool];
    __attribute__((aligned(16))) uint32_t stage_mult[kStageRows];
    int32_t stage[kStageRows][kHeadDim];
    __attribute__((aligned(16))) int32_t stage_z[kStageRows];
    // The ordered pass: its rows (tokens, or stretches as kSumRow | index), and
    // per half of the staging rows the largest bounds of its sums (kNoBound
    // without any) and whether it holds a special token.
    uint16_t order[kExactMaxTokens + kMaxBlocks + 8];
    float round_bound[2][kGroupsPerHead];
    uint32_t round_special[2];
    uint32_t staged;                              // rows taken so far
    uint32_t unbounded;                           // a sum could saturate Y
    // Special (first or rescaling) tokens of a split that cannot fold its own
    // sums; number i uses pool entry kPool-1-i for the ordinary tokens after
    // it in its block.  Per hot block: its first special token and their count.
    int8_t code[kSpecials][kHeadDim];
    uint32_t sp_word[kSpecials];
    uint32_t sp_exps[kSpecials];
    uint32_t hot_first[kPool];
    uint32_t hot_count[kPool];
    int32_t blk_max[kMaxBlocks];                  // per block: its largest score
    int32_t blk_exp[kMaxBlocks];                  // and the largest biased exponent of its V scales
    uint32_t limb_hi[2][kHeadDim / 4];            // query limbs 3 and 4
    uint32_t lut[33];
    int8_t new_code[kHeadDim];                    // the new token
    uint32_t new_exps;
    int32_t new_score;
    uint32_t specials;                            // special tokens so far
    int32_t prefix;                               // running maximum before the range
    uint32_t failed;                              // the range's sums are incomplete
    uint32_t z;                                   // Z over the range
    uint32_t new_word;                            // the new token's coefficient word
    uint32_t last;
    uint32_t misc[16];                            // the split's own maximum, count and words of entries 0 and 1
    uint32_t fail_at[2];                          // per folding wave: the first split whose sums cannot be used
    int32_t max_before[kExactMaxSplits];          // running maximum before each split
    int16_t q14[kHeadDim];
};

struct KBlock {
    v4i k[kRows];
    v2u s[kRows];
};
struct VBlock {
    v4i v[kRows];
};

// The page through one buffer resource: per-lane offsets fixed, the token
// offset in an SGPR.  `past` puts a load past the page's range (zeros, no
// memory access), for a wave without a (further) block.
struct Page {
    __amdgpu_buffer_rsrc_t rsrc;
    int32_t code_lane;       // lane's byte offset in a code plane
    int32_t scale_lane;      // lane's scale pair
    int32_t v_plane, s_plane, end;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t page_rsrc(int8_t* page, int cap) {
    return __builtin_amdgcn_make_buffer_rsrc(page, static_cast<short>(0), cap * kTokenBytes, kBufferWord3);
}
__device__ __forceinline__ Page make_page(__amdgpu_buffer_rsrc_t rsrc, int cap, int c, int r) {
    Page pg;
    pg.rsrc = rsrc;
    pg.code_lane = r * kCodeBytes + c * 16;
    pg.scale_lane = r * kScaleBytes + (c >> 1) * 8;
    pg.v_plane = cap * kCodeBytes;
    pg.s_plane = cap * 2 * kCodeBytes;
    pg.end = cap * kTokenBytes;
    return pg;
}

constexpr int kNontemporal = 2;

__device__ __forceinline__ void load_k_row(const Page& pg, int t, int32_t past, v4i& k, v2u& s) {
    k = __builtin_amdgcn_raw_buffer_load_b128(pg.rsrc, pg.code_lane + past, t * kCodeBytes, kNontemporal);
    s = __builtin_amdgcn_raw_buffer_load_b64(pg.rsrc, pg.scale_lane + past, pg.s_plane + t * kScaleBytes, kNontemporal);
}
__device__ __forceinline__ void load_v_row(const Page& pg, int t, int32_t past, v4i& v) {
    v = __builtin_amdgcn_raw_buffer_load_b128(pg.rsrc, pg.code_lane + past, pg.v_plane + t * kCodeBytes, kNontemporal);
}
__device__ __forceinline__ void load_k(const Page& pg, int t0, bool any, KBlock& kb) {
#pragma unroll
    for (int i = 0; i < kRows; ++i) load_k_row(pg, t0 + 8 * i, any ? 0 : pg.end, kb.k[i], kb.s[i]);
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void load_v(const Page& pg, int t0, bool any, VBlock& vb) {
#pragma unroll
    for (int i = 0; i < kRows; ++i) load_v_row(pg, t0 + 8 * i, any ? 0 : pg.end, vb.v[i]);
    __builtin_amdgcn_sched_barrier(0);
}

// Scores of a block, lane l getting token l's, and the exponents of its V
// scales; v_exp is the largest of those the lane holds.
// Three limbs and shifts up to 25 (every shift a quantized row has) keep each
// half-group's scaled dot below 2^49, so doubles hold it and the octet's sum
// exactly; the general form takes five limbs modulo 2^64.
__device__ __forceinline__ int32_t score_block(const KBlock& kb, const QueryLimbs& ql, bool q3, const Shared& sh,
                                               uint2* tok, int c, int r, int lane, int32_t& v_exp) {
    double own_f = 0.0;
    int64_t own_i = 0;
    uint32_t general = 0, vs = 0;      // pairs of rows in the general form; largest V scale
#pragma unroll
    for (int i = 0; i < kRows; i += 2) {
        if ((c & 1) == 0) {
            reinterpret_cast<uint8_t*>(&tok[8 * i + r].y)[c >> 1] = static_cast<uint8_t>(kb.s[i].y >> 23);
            reinterpret_cast<uint8_t*>(&tok[8 * i + 8 + r].y)[c >> 1] = static_cast<uint8_t>(kb.s[i + 1].y >> 23);
        }
        vs = max(vs, max(kb.s[i].y, kb.s[i + 1].y));
        if (q3 && __builtin_amdgcn_ballot_w64(max(kb.s[i].x, kb.s[i + 1].x) >= (136u << 23)) == 0) {
            double t[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const double f = static_cast<double>(__uint_as_float(kb.s[i + u].x));   // 2^(shift-17)
                t[u] = octet_sum_f64(__builtin_floor(limb_dot3(ql, kb.k[i + u]) * f * 128.0));
            }
            if (c == i) own_f = t[0];
            if (c == i + 1) own_f = t[1];
        } else {
            general |= 3u << i;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                int32_t a3 = 0, a4 = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    a3 = __builtin_amdgcn_sdot4(static_cast<int32_t>(sh.limb_hi[0][4 * c + j]), kb.k[i + u][j], a3, false);
                    a4 = __builtin_amdgcn_sdot4(static_cast<int32_t>(sh.limb_hi[1][4 * c + j]), kb.k[i + u][j], a4, false);
                }
                const int64_t s = static_cast<int64_t>(limb_dot3(ql, kb.k[i + u])) + (static_cast<int64_t>(a3) << 24) +
                                  (static_cast<int64_t>(a4) << 32);
                const int64_t t = octet_sum64(scaled_half(s, shift_of(__uint_as_float(kb.s[i + u].x))));
                if (c == i + u) own_i = t;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    v_exp = static_cast<int32_t>(vs >> 23);
    const int32_t score = score_of((general >> c) & 1u ? own_i : static_cast<int64_t>(own_f));   // of token 8 c + r
    return __shfl(score, 8 * (lane & 7) + (lane >> 3));
}

// The scores of block `blk` of the range [first, end) into its tokens, and its
// largest score and V scale; whether it has a V shift of 16 or more.
__device__ __forceinline__ bool take_scores(const KBlock& kb, const QueryLimbs& ql, bool q3, Shared& sh, int blk,
                                            int first, int end, int c, int r, int lane) {
    uint2* const tok = sh.tok + blk * kBlock;
    int32_t v_exp;
    const int32_t score = score_block(kb, ql, q3, sh, tok, c, r, lane, v_exp);
    tok[lane].x = static_cast<uint32_t>(score);
    const int32_t mx = wave_scan_max(first + blk * kBlock + lane < end ? score : INT32_MIN);
    v_exp = wave_scan_max(v_exp);
    if (lane == 63) {
        sh.blk_max[blk] = mx;
        sh.blk_exp[blk] = v_exp;
    }
    return __builtin_amdgcn_readlane(v_exp, 63) >= static_cast<int32_t>(__float_as_uint(kWideScale) >> 23);
}

// The coefficient words of a block's tokens (lane = token) from their scores;
// `start` is the running maximum before the block, which holds a new one if
// is_hot.
__device__ __forceinline__ uint32_t take_words(Shared& sh, int blk, int first, int end, int32_t start, bool is_hot,
                                               int lane) {
    uint2* const tok = sh.tok + blk * kBlock;
    const bool valid = first + blk * kBlock + lane < end;
    const int32_t score = static_cast<int32_t>(tok[lane].x);
    int32_t pm = start;                            // running maximum before the lane's token
    if (is_hot) {
        pm = dpp_shifted<kDppWaveShr1, 0xF>(INT32_MIN, wave_scan_max(valid ? score : INT32_MIN));
        pm = lane == 0 ? start : max(pm, start);
    }
    const bool init = first + blk + lane == 0;
    const uint32_t word = !valid ? 0u : init ? kInit : coef_word(score, pm, sh.lut);
    tok[lane].x = __float_as_uint(static_cast<float>(word & kCoefMask)) |
                  ((word & (kInit | kRescale)) != 0u ? 0x80000000u : 0u);
    wave_lds_sync();
    return word;
}

// A wave's running sums of ordinary terms: per lane 16 channels of chunk c
// over rows r, r + 8, ... of its blocks.
struct Sums {
    uint32_t acc[16];
    float bound;             // sum of the p of the lane's group
    uint32_t z;              // coefficients of the lane's own tokens (lane = token)
    uint32_t rows;           // terms added per channel (each carries kRoundMagicBits)
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j] = 0u;
        bound = 0.0f;
        z = rows = 0u;
    }
};

// Sums stand here, and no load moves across: left alone, the compiler adds a
// block's terms as one tree, holding all of them, and loads every row first.
__device__ __forceinline__ void pin(uint32_t* x) {
    asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]), "+v"(x[6]), "+v"(x[7]),
                      "+v"(x[8]), "+v"(x[9]), "+v"(x[10]), "+v"(x[11]), "+v"(x[12]), "+v"(x[13]), "+v"(x[14]),
                      "+v"(x[15])
                 :
                 : "memory");
}

// The product p of the lane's coefficient and its group's V scale (exact).
__device__ __forceinline__ float token_product(uint2 w, uint32_t rot) {
    return __uint_as_float(w.x) * __uint_as_float(__builtin_amdgcn_alignbit(w.y, w.y, rot) & 0x7f800000u);
}

// Adds the terms of the block's tokens [a, b) (all of them unless MASKED).
// Two rows at a time, so that one three-operand add takes both terms.
template <bool MASKED>
__device__ __forceinline__ void add_terms(const VBlock& vb, const uint2* tok, int r, uint32_t rot, int a, int b,
                                          Sums& s) {
    uint2 w[kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i) w[i] = tok[8 * i + r];
#pragma unroll
    for (int i = 0; i < kRows; i += 2) {
        if (!MASKED || (8 * i + 16 > a && 8 * i < b)) {
            float p[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int t = 8 * (i + u) + r;
                p[u] = token_product(w[i + u], rot);
                if (MASKED && (t < a || t >= b)) p[u] = 0.0f;
                s.bound += p[u];
            }
            s.rows += 2;
            v4i v0 = vb.v[i], v1 = vb.v[i + 1];
            if (MASKED) asm volatile("" : "+v"(v0), "+v"(v1));   // as in add_wide_terms
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int32_t c0 = static_cast<int8_t>(v0[j >> 2] >> (8 * (j & 3)));
                const int32_t c1 = static_cast<int8_t>(v1[j >> 2] >> (8 * (j & 3)));
                s.acc[j] += term_bits(c0, p[0]) + term_bits(c1, p[1]);
            }
            pin(s.acc);
        }
    }
}

// The terms of a block with a V shift of 16 or more.  code p is exact in FP32
// (at most 24 significant bits), so rint rounds it to nearest even; shifts of
// 24 and more, whose terms may leave the int32 range, make the bound infinite.
// The empty asm keeps the compiler from sharing the conversions with the other
// form: hoisted above the choice between them they would hold 128 registers.
__device__ __forceinline__ void add_wide_terms(VBlock& vb, const uint2* tok, int r, uint32_t rot, int a, int b,
                                               Sums& s) {
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        const int t = 8 * i + r;
        const uint2 w = tok[t];
        const float p = t >= a && t < b ? token_product(w, rot) : 0.0f;
        s.bound += p;
        if ((__builtin_amdgcn_alignbit(w.y, w.y, rot) & 0x7f800000u) >= __float_as_uint(kHugeScale)) s.bound = INFINITY;
        v4i v = vb.v[i];
        asm volatile("" : "+v"(v));
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int32_t code = static_cast<int8_t>(v[j >> 2] >> (8 * (j & 3)));
            s.acc[j] += static_cast<uint32_t>(static_cast<int32_t>(__builtin_rintf(static_cast<float>(code) * p)));
        }
        pin(s.acc);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Adds a wave's sums to pool entry e and clears them.  The 16 channels' sums
// over 8 rows reduce by halves: two permlane swaps pair the rows of the upper
// and lower half-waves and of the odd and even 16-lane rows while the channels
// spread over them, and a rotation adds the last pair.
__device__ __forceinline__ void flush(Shared& sh, int e, Sums& s, int lane) {
    asm volatile("" : "+v"(lane));   // keeps the addresses below out of registers across the loop around the call
    const uint32_t magic = s.rows * kRoundMagicBits;
    uint32_t h8[8], h4[4];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const auto x = __builtin_amdgcn_permlane32_swap(s.acc[j] - magic, s.acc[j + 8] - magic, false, false);
        h8[j] = x[0] + x[1];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const auto x = __builtin_amdgcn_permlane16_swap(h8[j], h8[j + 4], false, false);
        h4[j] = x[0] + x[1];
        h4[j] += dpp_u<kDppRowRor8>(h4[j]);
    }
    // lane: channels 8 (lane >> 5) + 4 ((lane >> 4) & 1) + 0..3 of chunk c, two of them per bit 3
    const int c = lane & 7, up = (lane >> 3) & 1;
    const int ch = 16 * c + 8 * (lane >> 5) + 4 * ((lane >> 4) & 1) + 2 * up;
    atomicAdd(reinterpret_cast<uint32_t*>(&sh.pool[e][ch]), up ? h4[2] : h4[0]);
    atomicAdd(reinterpret_cast<uint32_t*>(&sh.pool[e][ch + 1]), up ? h4[3] : h4[1]);
    const float bound = across_octets_sum(s.bound);
    if ((lane & 7) == lane && (lane & 1) == 0) atomicAdd(&sh.pool_b[e][lane >> 1], bound);
    const uint32_t z = wave_scan_add(s.z);
    if (lane == 63) atomicAdd(&sh.pool_z[e], z);
    s.clear();
}

// Where |y| plus the bound of a segment's terms stays below 2^31 no partial
// sum saturates.  The bound: |code| <= 128, half a unit of rounding per term
// and the roundings of the float sums.
constexpr float kReach = 2147483000.0f;
__device__ __forceinline__ float bound_reach(float b) { return b * 128.125f + 8192.0f; }
__device__ __forceinline__ bool bounded(int32_t y, float b) {
    return __builtin_fabsf(static_cast<float>(y)) + bound_reach(b) < kReach;
}

__device__ __forceinline__ uint32_t exps_shift(uint32_t exps, int g) { return ((exps >> (8 * g)) & 0xffu) - 110u; }
__device__ __forceinline__ uint32_t token_coef(uint32_t x) {
    return static_cast<uint32_t>(__builtin_fabsf(__uint_as_float(x)));
}

// Word of channel d in a staging row.  A lane writes 16 channels, four words at
// a time: quad q of chunk c goes to word 4 (8 q + (c ^ 2 q)), so that eight
// lanes write 128 bytes in a row (16 c + 4 q has four of them on each bank) and
// the 32 channels of half a wave read from 32 banks.
__device__ __forceinline__ int stage_quad(int c, int q) { return 4 * (8 * q + (c ^ (2 * q))); }
__device__ __forceinline__ int stage_column(int d) { return stage_quad((d >> 4) & 7, (d >> 2) & 3) + (d & 3); }

// Stages a token's terms for 16 channels: v itself for a special token (its
// 2^17 scale = 2^shift), else the rounded product.  As the largest shift among
// the tokens allows: one fused multiply-add (up to 15), a product and rint (up
// to 23), 64-bit integers.
enum TermForm { kTermFma, kTermRint, kTermAny };
template <TermForm FORM>
__device__ __forceinline__ void stage_row(int32_t* row, int c, v4i v, uint2 w, uint32_t rot) {
    const uint32_t scale = __builtin_amdgcn_alignbit(w.y, w.y, rot) & 0x7f800000u;
    const bool special = (w.x >> 31) != 0u;
    if constexpr (FORM == kTermAny) {
        const uint32_t coef = special ? 1u << 17 : token_coef(w.x);
#pragma unroll 1
        for (int q = 0; q < 4; ++q) {
            v4i x;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                x[j] = mulq17_wrap(dequant_raw(static_cast<int8_t>(v[0] >> (8 * j)), (scale >> 23) - 110u), coef);
            *reinterpret_cast<v4i*>(row + stage_quad(c, q)) = x;
            v = __builtin_shufflevector(v, v, 1, 2, 3, 0);
        }
    } else {
        const float p = (special ? 131072.0f : __uint_as_float(w.x)) * __uint_as_float(scale);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v4i x;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int32_t code = static_cast<int8_t>(v[q] >> (8 * j));
                x[j] = FORM == kTermFma ? static_cast<int32_t>(term_bits(code, p) - kRoundMagicBits)
                                        : static_cast<int32_t>(__builtin_rintf(static_cast<float>(code) * p));
            }
            *reinterpret_cast<v4i*>(row + stage_quad(c, q)) = x;
        }
    }
}

// Y of a channel (its word `col` of a staging row), or Z (Z, every lane), over
// `rows` (at most 64) staged tokens from row `at`.
template <bool Z>
__device__ __forceinline__ int32_t run_staged(const Shared& sh, uint32_t at, int rows, int col, int lane, int32_t y) {
    constexpr int kAhead = 8;
    const uint32_t mult = lane < rows ? sh.stage_mult[at + static_cast<uint32_t>(lane)] : 1u << 17;
    const uint64_t special = __builtin_amdgcn_ballot_w64(mult != 1u << 17);
    int32_t next[kAhead];
    auto load = [&](int r) {
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            const uint32_t row = at + static_cast<uint32_t>(min(r + j, rows - 1));
            next[j] = Z ? sh.stage_z[row] : sh.stage[row][col];
        }
    };
    load(0);
    for (int r = 0; r < rows; r += kAhead) {
        int32_t term[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) term[j] = r + j < rows ? next[j] : 0;
        load(r + kAhead);
        const uint32_t sp = static_cast<uint32_t>(special >> r) & 0xffu;
        if (sp == 0u) {
#pragma unroll
            for (int j = 0; j < kAhead; ++j) y = __builtin_elementwise_add_sat(y, term[j]);
        } else {
#pragma unroll
            for (int j = 0; j < kAhead; ++j) {
                if ((sp >> j) & 1u)
                    y = mulq17_wrap(y, static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(mult), r + j)));
                y = __builtin_elementwise_add_sat(y, term[j]);
            }
        }
    }
    return y;
}

// The ordered pass: Y and Z token by token, all waves at it, where sums do not
// serve: hot blocks past the staging rows, stretches whose sum could saturate
// Y, splits with more special tokens than entries.  It runs over a list of
// rows, in rounds of 64: waves 4 to 7 gather the V codes of the rows' tokens
// from the page, four rounds ahead, and stage their terms in one half of the
// staging rows, and wave 3 what else the rows have; waves 0 and 1 take Y and
// wave 2 takes Z over the other half.  LDS and the instructions of both sides
// bound a round together: 0.7 us where every token adds a term, 1.25 where every
// token rescales (0.3 the staging alone, 0.35 and 0.85 the fold alone).
constexpr int kRound = kStageRows / 2;
constexpr int kFetchAhead = 4;
constexpr int kSumRow = 0x8000;
constexpr float kNoBound = -1e9f;                 // of a row that is no sum

// Y (or Z) over a staged round's rows from row `at` (those past the list's end
// add nothing): sat32(RNE(Y m) + x).  A row goes through a double, three
// dependent operations: the product (50 bits) plus 1.5 2^52 rounds once, to an
// integer, to nearest even, and the low word is that integer.  In a loop alone,
// from LDS: 13.3 ns a row; the 64-bit integer form 25.8, clamping in doubles
// 18.8, rint and convert 16.7.  One straight path for the round: chosen every 8
// rows, the taken branches cost more than the additions between them.
// `worst`: the largest |Y| around a round's sums, plus their largest bound.
template <bool Z>
__device__ __forceinline__ int32_t run_round(const Shared& sh, int at, int d, int lane, int32_t y, float& worst) {
    const int g = (d >> 5) & 3, col = stage_column(d);
    int32_t x[kRound];
    auto load = [&](int r) {
#pragma unroll
        for (int j = r; j < r + kRound / 2; ++j)
            if (!Z) x[j] = sh.stage[at + j][col];
    };
    const int own = static_cast<int>(sh.stage_mult[at + lane]);   // of row `lane`
    const int own_z = Z ? sh.stage_z[at + lane] : 0;
    const uint32_t has_special = sh.round_special[at / kRound];
    const float bound = Z ? kNoBound : sh.round_bound[at / kRound][g];
    load(0);
    const bool special = uniform(has_special) != 0u;
    const bool sums = uniform(__float_as_int(bound)) != __float_as_int(kNoBound);
    load(kRound / 2);
    auto term = [&](int j) { return Z ? __builtin_amdgcn_readlane(own_z, j) : x[j]; };
    auto step = [&](int j) {
        const float m = __int_as_float(__builtin_amdgcn_readlane(own, j));
        const double t = __builtin_fma(static_cast<double>(y), static_cast<double>(m), 0x1.8p52);
        y = __builtin_elementwise_add_sat(static_cast<int32_t>(__double2loint(t)), term(j));
    };
    if (Z && !special) {   // Z stays below 2^30: a sum in any order
        y += __builtin_amdgcn_readlane(static_cast<int>(wave_scan_add(static_cast<uint32_t>(own_z))), 63);
    } else if (!sums && !special) {
#pragma unroll
        for (int j = 0; j < kRound; ++j) y = __builtin_elementwise_add_sat(y, term(j));
    } else if (!sums) {
#pragma unroll
        for (int j = 0; j < kRound; ++j) step(j);
    } else {
        int32_t hi = y, lo = y;
#pragma unroll
        for (int j = 0; j < kRound; ++j) {
            step(j);
            hi = max(hi, y);
            lo = min(lo, y);
        }
        const int32_t most = max(hi, lo == INT32_MIN ? INT32_MAX : -lo);
        worst = fmaxf(worst, static_cast<float>(most) + bound_reach(bound));
    }
    return y;
}

__device__ __forceinline__ int round_barriers(int rounds) {
    return (rounds + kFetchAhead - 1) / kFetchAhead * kFetchAhead;
}

// Waves 4 to 7: the terms of all rounds.
template <TermForm FORM, bool PIECES>
__device__ __forceinline__ void stage_rounds(__amdgpu_buffer_rsrc_t rsrc, Shared& sh, int cap, int first, int total,
                                             int rounds, int wave, int lane) {
    struct Fetched {
        v4i v[2];
        uint2 word[2];
        int sum[2];                               // a sum's index, or -1
    };
    Fetched f[kFetchAhead];
    const int c = lane & 7, mine = 8 * (wave - 4) + (lane >> 3);   // and 32 more
    const uint32_t rot = (9u + 8u * static_cast<uint32_t>(c >> 1)) & 31u;
    auto fetch = [&](int round, Fetched& x) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int i = round * kRound + mine + 32 * u;
            const int row = PIECES ? static_cast<int>(sh.order[min(i, total - 1)]) : i;
            const bool sum = PIECES && row >= kSumRow && i < total, none = sum || i >= total;
            const int token = none ? 0 : row;
            x.word[u] = sh.tok[none ? kExactMaxTokens : row];
            x.sum[u] = sum ? row & (kSumRow - 1) : -1;
            x.v[u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (first + token) * kCodeBytes + 16 * c, cap * kCodeBytes, 0);
        }
    };
    auto stage = [&](int round, const Fetched& x) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            int32_t* const to = sh.stage[(round & 1) * kRound + mine + 32 * u];
            stage_row<FORM>(to, c, x.v[u], x.word[u], rot);
            if (PIECES && x.sum[u] >= 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<v4i*>(to + stage_quad(c, q)) =
                        reinterpret_cast<const v4i*>(&sh.pool[x.sum[u]][16 * c])[q];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int u = 0; u < kFetchAhead; ++u) fetch(u, f[u]);
    stage(0, f[0]);
    fetch(kFetchAhead, f[0]);
    // Barrier b hands round b to the folding waves.  The fetches are made on
    // every path, so that the loads in flight stay countable.
    for (int b = 0; b < round_barriers(rounds); b += kFetchAhead) {
#pragma unroll
        for (int u = 0; u < kFetchAhead; ++u) {
            __syncthreads();
            const int round = b + u + 1;
            if (round < rounds) stage(round, f[(u + 1) % kFetchAhead]);
            fetch(round + kFetchAhead, f[(u + 1) % kFetchAhead]);
        }
    }
}

// With `pieces` its rows are the tokens of the hot blocks' spans, and in front
// of each span and after the last one the sum of the stretch there (where one
// fails its bound sh.unbounded is set); without, tokens [0, count).  `first` is
// the sequence position of token 0.  Returns Y (waves 0 and 1) or Z (wave 2)
// from `y`.  Every wave makes the same number of barriers.
//
// Out of line, so that its registers are its own: inlined, the kernel's own
// path spills, and took 26.0 us at batch 1 against 23.9.  Arguments arrive in vector registers; all but
// y are wave-uniform.
typedef __attribute__((address_space(3))) Shared* SharedPtr;
__device__ __attribute__((noinline)) int32_t ordered_pass(int8_t* page, SharedPtr shared, int cap_arg, int first_arg,
                                                          int count_arg, int pieces_arg, int nbound_arg, int32_t y) {
    Shared& sh = *(Shared*)shared;
    const int first = uniform(first_arg), count = uniform(count_arg);
    const int nbound = uniform(nbound_arg), cap = uniform(cap_arg);
    const bool pieces = uniform(pieces_arg) != 0;
    const __amdgpu_buffer_rsrc_t rsrc = page_rsrc(uniform(page), cap);
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, d = threadIdx.x;
    int total = count;
    if (pieces) {
        const uint32_t span = lane < nbound ? sh.hot[lane].x : 0u;
        const int32_t len = static_cast<int32_t>(span >> 16) - static_cast<int32_t>(span & 0xffffu);
        const int32_t past = static_cast<int32_t>(wave_scan_add(lane < nbound ? static_cast<uint32_t>(len) + 1u : 0u));
        total = __builtin_amdgcn_readlane(past, 63) + 1;
        for (int k = wave; k < nbound; k += kWaves) {
            const int n = __builtin_amdgcn_readlane(len, k), at = __builtin_amdgcn_readlane(past, k) - n;
            const int token = __builtin_amdgcn_readlane(static_cast<int>(span), k) & 0xffff;
            if (lane < n) sh.order[at + lane] = static_cast<uint16_t>(token + lane);
            if (lane == 0) sh.order[at - 1] = static_cast<uint16_t>(kSumRow | k);
        }
        if (d == 0) sh.order[total - 1] = static_cast<uint16_t>(kSumRow | nbound);
        __syncthreads();
    }
    const int rounds = (total + kRound - 1) / kRound;
    const int barriers = round_barriers(rounds);
    if (rounds == 0) return y;
    if (wave >= 4) {
        const int widest = __builtin_amdgcn_readlane(
            wave_scan_max(lane < (count + kBlock - 1) / kBlock ? sh.blk_exp[lane] : 0), 63);
        auto produce = [&](auto form) {
            if (pieces) stage_rounds<form.value, true>(rsrc, sh, cap, first, total, rounds, wave, lane);
            else stage_rounds<form.value, false>(rsrc, sh, cap, first, total, rounds, wave, lane);
        };
        if (widest >= static_cast<int>(__float_as_uint(kHugeScale) >> 23))
            produce(std::integral_constant<TermForm, kTermAny>());
        else if (widest >= static_cast<int>(__float_as_uint(kWideScale) >> 23))
            produce(std::integral_constant<TermForm, kTermRint>());
        else
            produce(std::integral_constant<TermForm, kTermFma>());
    } else if (wave == 3) {
        auto describe = [&](int round) {          // lane = row
            const int i = round * kRound + lane, at = (round & 1) * kRound + lane;
            const int row = pieces ? static_cast<int>(sh.order[min(i, total - 1)]) : i;
            const bool past = i >= total, sum = pieces && row >= kSumRow;
            const uint32_t x = past || sum ? 0u : sh.tok[row].x;
            const bool special = (x >> 31) != 0u;
            const float coef = __builtin_fabsf(__uint_as_float(x));
            float mult = special ? coef * 0x1p-17f : 1.0f;   // 0.0 for the sequence's first token
            int32_t z = special ? 1 << 17 : static_cast<int32_t>(coef);
            float4 bound = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (sum && !past) {
                z = static_cast<int32_t>(sh.pool_z[row & (kSumRow - 1)]);
                bound = *reinterpret_cast<const float4*>(sh.pool_b[row & (kSumRow - 1)]);
            }
            sh.stage_mult[at] = __float_as_uint(mult);
            sh.stage_z[at] = z;
            const uint64_t specials = __builtin_amdgcn_ballot_w64(special);
            if (pieces) {                         // the bounds are not negative: their bits compare as integers do
                const float b[kGroupsPerHead] = {bound.x, bound.y, bound.z, bound.w};
#pragma unroll
                for (int g = 0; g < kGroupsPerHead; ++g) {
                    const int32_t most = wave_scan_max(sum && !past ? __float_as_int(b[g]) : __float_as_int(kNoBound));
                    if (lane == 63) sh.round_bound[round & 1][g] = __int_as_float(most);
                }
            } else if (lane < kGroupsPerHead) {
                sh.round_bound[round & 1][lane] = kNoBound;
            }
            if (lane == 0) sh.round_special[round & 1] = specials != 0u;
        };
        describe(0);
        for (int b = 0; b < barriers; ++b) {
            __syncthreads();
            if (b + 1 < rounds) describe(b + 1);
        }
    } else {
        float worst = 0.0f;
        __builtin_amdgcn_s_setprio(3);             // ahead of the staging wave on its SIMD
        for (int b = 0; b < barriers; ++b) {
            __syncthreads();
            const int at = (b & 1) * kRound;
            if (b < rounds) {
                if (wave < 2) y = run_round<false>(sh, at, d, lane, y, worst);
                else y = run_round<true>(sh, at, d, lane, y, worst);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        if (!(worst < kReach)) sh.unbounded = 1u;
    }
    return y;
}

// Runs the head from token `first` on, in order, after the sums of the splits
// before: scores, coefficients (the new token's too), then the ordered pass
// from `y` (Y in waves 0 and 1, Z in wave 2).  Out of line like it.
__device__ __attribute__((noinline)) int32_t run_rest(int8_t* page, SharedPtr shared, int cap_arg, int first_arg,
                                                      int end_arg, int32_t max_before, v4i q0, v4i q1, v4i q2, int q3,
                                                      int32_t y) {
    Shared& sh = *(Shared*)shared;
    const int cap = uniform(cap_arg), first = uniform(first_arg), end = uniform(end_arg), count = end - first;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int c = lane & 7, r = lane >> 3;
    const Page pg = make_page(page_rsrc(uniform(page), cap), cap, c, r);
    const int blocks = (count + kBlock - 1) / kBlock;
    QueryLimbs ql;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        ql.w[0][j] = q0[j];
        ql.w[1][j] = q1[j];
        ql.w[2][j] = q2[j];
    }
    KBlock kb;
    load_k(pg, first + wave * kBlock, wave < blocks, kb);
    for (int blk = wave; blk < blocks; blk += kWaves) {
        (void)take_scores(kb, ql, uniform(q3) != 0, sh, blk, first, end, c, r, lane);
        load_k(pg, first + (blk + kWaves) * kBlock, blk + kWaves < blocks, kb);
    }
    __syncthreads();
    const int32_t m = max(max_before, wave_scan_max(lane < blocks ? sh.blk_max[lane] : INT32_MIN));
    int32_t before = dpp_shifted<kDppWaveShr1, 0xF>(INT32_MIN, m);
    before = lane == 0 ? max_before : before;
    for (int blk = wave; blk < blocks; blk += kWaves)
        (void)take_words(sh, blk, first, end, __builtin_amdgcn_readlane(before, blk), true, lane);
    if (wave == 0 && lane == 0) sh.new_word = coef_word(sh.new_score, __builtin_amdgcn_readlane(m, 63), sh.lut);
    __syncthreads();
    return ordered_pass(page, shared, cap, first, count, 0, 0, y);
}

// Tagged words of the split exchange: the launch's tag above a 32-bit value.
__device__ __forceinline__ void publish(uint64_t* p, uint32_t tag, uint32_t v) {
    __hip_atomic_store(p, (static_cast<uint64_t>(tag) << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t fetch(const uint64_t* p) {
    return __hip_atomic_load(const_cast<uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool current(uint64_t w, uint32_t tag) { return static_cast<uint32_t>(w >> 32) == tag; }

// Rounds of re-reads (about a microsecond each) a split waits for the maxima
// of the splits before it.  They are resident in every launch the plan makes
// on an idle GPU; where other work keeps one off it, the split gives up.
constexpr uint32_t kPrefixPolls = 256;

// A split's slot: its maximum, then its entries.  Entry e holds the sums
// A[128], the values V[128] of the special token they follow (none for entry
// 0), and six words {z, word, bounds of the four groups}; those of entries 0
// and 1 lie together behind the maximum and the count, so that one load per
// split, a word per lane, takes all of them.
constexpr uint32_t kSlotFailed = 1u << 31;
constexpr int kSlotMax = 0, kSlotCount = 1, kSlotMisc = 2, kSlotEntries = kSlotMisc + 6 * kExactEntries;
static_assert(kExactSlotWords >= kSlotEntries + kExactEntries * 2 * kHeadDim, "slot layout");
__device__ __forceinline__ uint64_t* slot_misc(uint64_t* slot, int e) { return slot + kSlotMisc + 6 * e; }
__device__ __forceinline__ uint64_t* slot_sums(uint64_t* slot, int e) { return slot + kSlotEntries + e * 2 * kHeadDim; }
__device__ __forceinline__ uint64_t* slot_values(uint64_t* slot, int e) { return slot_sums(slot, e) + kHeadDim; }

// Argument-block fields used late, loaded while the first blocks are in flight.
struct Tail {
    int32_t* out;
    uint8_t* act_q;
    uint8_t* act_scale;
    uint32_t merge_polls;
    uint32_t merge_tag_skew;
};

template <bool Q17, bool SPLIT>
__global__ __launch_bounds__(kThreads) void exact_kernel(const int8_t* layer_pages, uint32_t geometry,
                                                         uint32_t dispatch, const void* q_in, const void* k_in,
                                                         const void* v_in, const int2* lut, const void* aux,
                                                         StepArgs a) {
    constexpr int kIn = Q17 ? kInQ17 : kInF32;
    __shared__ Shared sh;
    const uint32_t uniform_pos = dispatch & StepPreload::kRowsListed;
    auto row_of = [&](int z) {
        return uniform_pos != StepPreload::kRowsListed ? pack_row(z, uniform_pos) : a.rows[z];
    };
    // The upper half of `dispatch`: the split's tokens when SPLIT, else the rows
    // less one and a 32nd of the workgroups (the argument block and the grid's
    // size are a scalar round trip to host memory away).
    const int C = static_cast<int>(dispatch >> 16) * kSplitQuantum;
    const int heads = static_cast<int>((dispatch >> 16 & 0xffu) + 1u) * kHeads;
    const int stride = static_cast<int>(dispatch >> 24) * kHeads;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    int lane = threadIdx.x & 63, d = threadIdx.x;
    int c = lane & 7, r = lane >> 3;
    const int cap = static_cast<int>(geometry & 0xffffu);
    const int split = SPLIT ? blockIdx.x : 0;

    // The head in work.  [begin, stop) are its cached tokens of this
    // workgroup; the new token is the last step.
    uint32_t row = SPLIT ? row_of(blockIdx.z) : row_of(blockIdx.x / kHeads);
    int h = SPLIT ? blockIdx.y : blockIdx.x % kHeads;
    int b = static_cast<int>(row & 0xffu), pos = static_cast<int>(row >> 8);
    if (SPLIT && split * C > pos) return;
    const int nsplit = SPLIT ? (pos + C) / C : 1;
    const bool owner = split == nsplit - 1;       // appends the new row
    const bool whole = nsplit == 1;
    const int begin = split * C;
    auto page_of = [&](int seq, int head) {
        return const_cast<int8_t*>(layer_pages) + (static_cast<int64_t>(seq) * (geometry >> 16) * kHeads + head) *
                                                      (static_cast<int64_t>(cap) * kTokenBytes);
    };
    Page pg = make_page(page_rsrc(page_of(b, h), cap), cap, c, r);

    // All loads of the prologue, then the first K and V blocks, before any math.
    int2 cs;
    InPair<kIn> row_q, row_k{}, row_v{};
    auto blocks_of = [&](int position) {           // blocks of the range
        return ((SPLIT ? min(C, position - begin) : position) + kBlock - 1) / kBlock;
    };
    auto load_inputs = [&](int seq, int head, int position) {
        const size_t row_elem = static_cast<size_t>(seq) * kModelDim + head * kHeadDim + 2 * lane;
        cs = lut[static_cast<size_t>(position) * kRopePairs + lane];
        row_q = load_in<kIn>(q_in, row_elem, 0);
        if (wave == kWaves - 1) {
            row_k = load_in<kIn>(k_in, row_elem, 0);
            row_v = load_in<kIn>(v_in, row_elem, 0);
        }
    };
    uint64_t* const workspace = static_cast<uint64_t*>(const_cast<void*>(aux));
    uint64_t* const arrival = workspace + kExactTableWords + (static_cast<size_t>(b) * kHeads + h) * kArrivalStride;
    load_inputs(b, h, pos);
    KBlock kb;
    VBlock vb;
    load_k(pg, begin + wave * kBlock, wave < blocks_of(pos), kb);
    load_v(pg, begin + wave * kBlock, wave < blocks_of(pos), vb);
    const uint64_t arrival_word = SPLIT ? fetch(arrival) : 0u;
    const uint32_t exp_entry = reinterpret_cast<const uint32_t*>(workspace)[lane];
    const Tail tail{reinterpret_cast<int32_t*>(a.out), a.act_q, a.act_scale, a.merge_polls, a.merge_tag_skew};
    __builtin_amdgcn_sched_barrier(0);

    for (int turn = 1;; ++turn) {
    // Derived per turn: what depends on the lane alone would otherwise stand in
    // registers through the whole loop, hundreds of addresses.
    asm volatile("" : "+v"(lane), "+v"(d));
    c = lane & 7;
    r = lane >> 3;
    pg.code_lane = r * kCodeBytes + c * 16;
    pg.scale_lane = r * kScaleBytes + (c >> 1) * 8;
    const int stop = SPLIT ? min(begin + C, pos) : pos;
    const int nblk = blocks_of(pos), own_blocks = wave < nblk ? (nblk - wave + kWaves - 1) / kWaves : 0;
    // The next head: its first blocks are loaded behind this one's last.
    int next_b = b, next_h = h, next_pos = 0;
    bool more = false;
    if constexpr (!SPLIT) {
        const int slot = static_cast<int>(blockIdx.x);
        const int index = turn * stride + ((turn & 1) ? stride - 1 - slot : slot);
        more = index < heads;
        if (more) {
            const uint32_t row = row_of(index / kHeads);
            next_h = index % kHeads;
            next_b = static_cast<int>(row & 0xffu);
            next_pos = static_cast<int>(row >> 8);
        }
    }
    Page next = pg;
    next.rsrc = page_rsrc(page_of(next_b, next_h), cap);
    const int32_t next_past = more && wave < blocks_of(next_pos) ? 0 : pg.end;
    for (int i = d; i < kPool * kHeadDim / 4; i += kThreads)
        reinterpret_cast<int4*>(&sh.pool[0][0])[i] = make_int4(0, 0, 0, 0);
    if (d < kPool) {
        sh.pool_z[d] = 0u;
        *reinterpret_cast<float4*>(sh.pool_b[d]) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    if (d == 0) {
        sh.tok[kExactMaxTokens] = make_uint2(0u, 0u);
        sh.specials = 0u;
        sh.staged = 0u;
        sh.unbounded = 0u;
        sh.failed = 0u;
    }

    // Query limbs: lane l splits channels 2l, 2l+1; each lane gathers limbs
    // 0-2 of its chunk.  limb k+1 = (what limb k leaves) / 256, which is the
    // arithmetic shift plus limb k's sign bit.
    QueryLimbs ql;
    bool q3;
    {
        const int2 qi = in_to_q17<kIn>(row_q);
        int32_t q[2];
        rope_pair(qi.x, qi.y, cs, q[0], q[1]);
        uint32_t half[5] = {0u, 0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            int32_t rest = q[i];
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                half[k] |= (static_cast<uint32_t>(rest) & 0xffu) << (8 * i);
                rest = (rest >> 8) + ((rest >> 7) & 1);
            }
        }
        q3 = __builtin_amdgcn_ballot_w64((half[3] | half[4]) != 0u) == 0;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const uint32_t dword = half[k] | (dpp_u<kDppQuadXor1>(half[k]) << 16);   // valid at even lanes
            if (k < 3) {
#pragma unroll
                for (int j = 0; j < 4; ++j) ql.w[k][j] = static_cast<int32_t>(__shfl(dword, 8 * c + 2 * j));
            } else if ((lane & 1) == 0) {
                sh.limb_hi[k - 3][lane >> 1] = dword;   // every wave writes the same words
            }
        }
        if (wave == kWaves - 1) {
            // The new row: codes and shifts, its score, and the append.
            const int2 ki = in_to_q17<kIn>(row_k), vi = in_to_q17<kIn>(row_v);
            int32_t k0, k1;
            rope_pair(ki.x, ki.y, cs, k0, k1);
            const RowCodes rc = row_codes(k0, k1, vi.x, vi.y);
            int64_t dot = static_cast<int64_t>(q[0]) * static_cast<int8_t>(rc.k0) +
                          static_cast<int64_t>(q[1]) * static_cast<int8_t>(rc.k1);
            dot = scaled_half(octet_sum64(dot), rc.sk);
#pragma unroll
            for (int s = 8; s < 64; s <<= 1) dot += __shfl_xor(dot, s);
            reinterpret_cast<uint16_t*>(sh.new_code)[lane] = static_cast<uint16_t>(rc.v0 | (rc.v1 << 8));
            if ((lane & 15) == 0) reinterpret_cast<uint8_t*>(&sh.new_exps)[lane >> 4] = static_cast<uint8_t>(rc.sv + 110u);
            if (lane == 0) sh.new_score = score_of(dot);
            if (owner) store_row(pg.rsrc, cap, pos, lane, rc);
        }
    }
    if (more) load_inputs(next_b, next_h, next_pos);

    // K pass.  Rows past `stop` are read (inside the page, or zero) and their
    // scores dropped.
    uint32_t wide_blocks = 0;                      // own blocks with a V shift of 16 or more
    // (One place loads the blocks, also for a wave without any: with several
    // the compiler gives them different registers, and copying between those
    // waits for the loads.)
    for (int it = 0; it == 0 || it < own_blocks; ++it) {
        if (own_blocks > 0 && take_scores(kb, ql, q3, sh, wave + it * kWaves, begin, stop, c, r, lane)) wide_blocks |= 1u << it;
        const bool here = it + 1 < own_blocks;
        load_k(here ? pg : next, here ? begin + (wave + (it + 1) * kWaves) * kBlock : wave * kBlock,
               here || next_past == 0, kb);
    }
    if (turn == 1 && d < 33) sh.lut[d] = exp_entry;
    asm volatile("" ::"s"(tail.out), "s"(tail.act_q), "s"(tail.act_scale), "s"(tail.merge_polls), "s"(tail.merge_tag_skew));
    __syncthreads();

    // The running maximum before every block (lane = block).
    const int32_t bm = lane < nblk ? sh.blk_max[lane] : INT32_MIN;
    const int32_t incl = wave_scan_max(bm);
    // Both halves of the word keep their registers until here: a register the
    // compiler reuses early waits for the load that still fills it.
    if (SPLIT) asm volatile("" ::"v"(arrival_word));
    const uint32_t tag = static_cast<uint32_t>(arrival_word >> 32) + 1u;
    const uint32_t want = tag + tail.merge_tag_skew;
    uint64_t* const slots =
        workspace + kExactTableWords + kExactArrivalWords + (exact_first_slot(b) * kHeads + h * exact_row_slots(b)) * static_cast<size_t>(kExactSlotWords);
    uint64_t* const mine = slots + split * kExactSlotWords;
    int32_t before_range = INT32_MIN;
    if (SPLIT && !whole) {
        if (wave == 0) {
            if (lane == 63) {
                publish(mine + kSlotMax, tag, static_cast<uint32_t>(incl));
                sh.misc[0] = static_cast<uint32_t>(incl);
            }
            int32_t m = INT32_MIN;
            bool ok = true;
            if (lane < split) {
                const uint64_t* p = slots + lane * kExactSlotWords + kSlotMax;
                uint64_t w = fetch(p);
                for (uint32_t n = 0; !current(w, want); ++n) {
                    if (n >= min(kPrefixPolls, tail.merge_polls)) {
                        ok = false;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                    w = fetch(p);
                }
                m = static_cast<int32_t>(static_cast<uint32_t>(w));
            }
            m = wave_scan_max(m);
            if (lane == 63) sh.prefix = m;
            if (!ok) sh.failed = 1u;
        }
        __syncthreads();
        before_range = uniform(sh.prefix);
    }
    int32_t before = dpp_shifted<kDppWaveShr1, 0xF>(INT32_MIN, incl);
    before = lane == 0 ? before_range : max(before, before_range);
    const uint64_t hot = __builtin_amdgcn_ballot_w64(lane < nblk && (bm > before || (begin == 0 && lane == 0)));
    // A stretch whose sum could saturate Y as far as its bound tells sends the
    // range through the ordered pass, so where coefficients stay near 1.0 over
    // many tokens of large V the stretches are cut, so that the bound of each
    // stays near 2^30.  Lane = block: 64 terms of at most 128 2^shift times the
    // largest coefficient, and the cuts where their running sum passes multiples
    // of 2^30.  (Batch 32, 4096 tokens, V scaled per token by e^(1.5 N(0, 1)):
    // 262 us; with a cut at every block where eight could pass 2^30, 279.)
    uint64_t cuts = 0;
    {
        const float coef = fast_exp2((static_cast<float>(min(bm, before)) - static_cast<float>(before)) *
                                     (1.4426950408889634f * 0x1p-17f));
        const float most = lane < nblk ? ldexpf(coef, sh.blk_exp[lane] - 110 + 13) : 0.0f;
        const int32_t passed = static_cast<int32_t>(fminf(wave_scan_add(most) * 0x1p-30f, 1e6f));
        cuts = __builtin_amdgcn_ballot_w64(lane > 0 && lane < nblk && passed != dpp_shifted<kDppWaveShr1, 0xF>(0, passed));
    }
    const uint64_t bounds = hot | cuts;            // where stretches end
    const int nbound = __builtin_popcountll(bounds);
    const int32_t top = max(before_range, __builtin_amdgcn_readlane(incl, 63));   // running maximum before the new token
    // Whether the fold can start at the range's first token: a hot block is
    // then run in order from its terms (staged in LDS as far as they fit);
    // other splits sum the pieces between its special tokens.
    const bool folds = !SPLIT || split == 0;
    static_assert(kMaxBlocks + 1 + kSpecials <= kPool, "an accumulator per stretch and per special token");

    // V pass.  First the coefficient words of a block's tokens.
    const uint32_t rot = (9u + 8u * static_cast<uint32_t>(c >> 1)) & 31u;   // exponent byte c / 2 to bits 23..30
    Sums s;
    s.clear();
    int stretch = 0;                               // hot blocks before the sums in hand
    bool dirty = false;
    for (int it = 0; it == 0 || it < own_blocks; ++it) {
    if (own_blocks > 0) {
        // The stretch the block's first tokens belong to: after the bound at
        // its start, if that is a cut, before it if the block is hot.
        const int blk = wave + it * kWaves;
        const bool is_hot = (hot >> blk) & 1ull, is_cut = !is_hot && ((cuts >> blk) & 1ull) != 0u;
        int k = __builtin_popcountll(bounds & ((1ull << blk) - 1ull));
        if (is_cut) {
            if (folds && lane == 0) sh.hot[k] = make_uint4(static_cast<uint32_t>(blk * kBlock) * 0x10001u, 0u, 0u, 0u);
            if (!folds && lane == 0) sh.hot_count[k] = 0u;
            ++k;
        }
        if (k != stretch && dirty) {
            flush(sh, stretch, s, lane);
            dirty = false;
        }
        stretch = k;
        const bool wide = (wide_blocks >> it) & 1u;
        const uint2* const tok = sh.tok + blk * kBlock;
        const uint32_t word = take_words(sh, blk, begin, stop, __builtin_amdgcn_readlane(before, blk), is_hot, lane);
        const uint32_t coef = word & kCoefMask;
        if (!is_hot) {
            s.z += coef;
            if (!wide) add_terms<false>(vb, tok, r, rot, 0, kBlock, s);
            else add_wide_terms(vb, tok, r, rot, 0, kBlock, s);
            dirty = true;
        } else if (folds) {
            // From the first to the last special token the block is run in
            // order later (by the ordered pass, where one block does not fit the
            // staging rows); the tokens before join the stretch that ends
            // here, those after the next one.
            const uint64_t m = __builtin_amdgcn_ballot_w64((word & (kInit | kRescale)) != 0u);
            const int t_first = __builtin_ctzll(m), t_last = 63 - __builtin_clzll(m);
            const int rows = t_last - t_first + 1;
            const uint2 own = tok[lane];
            const bool special = (own.x >> 31) != 0u;
            const uint32_t widest = max(max(own.y & 0xffu, (own.y >> 8) & 0xffu), max((own.y >> 16) & 0xffu, own.y >> 24));
            const bool huge = __builtin_amdgcn_ballot_w64(widest >= __float_as_uint(kHugeScale) >> 23) != 0;
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(&sh.staged, huge ? kStageRows + 1u : static_cast<uint32_t>(rows));
            at = uniform(at);
            if (lane == t_first)
                sh.hot[k] = make_uint4(static_cast<uint32_t>(blk * kBlock + t_first) |
                                           static_cast<uint32_t>(blk * kBlock + t_last + 1) << 16,
                                       at, (word & kInit) ? 0u : coef, 0u);
            if (!huge && at + static_cast<uint32_t>(rows) <= static_cast<uint32_t>(kStageRows)) {
                if (lane >= t_first && lane <= t_last) {
                    const uint32_t i = at + static_cast<uint32_t>(lane - t_first);
                    sh.stage_mult[i] = !special ? 1u << 17 : (word & kInit) ? 0u : coef;
                    sh.stage_z[i] = special ? 1 << 17 : static_cast<int32_t>(coef);
                }
#pragma unroll
                for (int i = 0; i < kRows; ++i) {
                    const int t = 8 * i + r;
                    v4i v = vb.v[i];
                    asm volatile("" : "+v"(v));   // as in add_wide_terms
                    if (t >= t_first && t <= t_last)
                        stage_row<kTermRint>(sh.stage[at + static_cast<uint32_t>(t - t_first)], c, v, tok[t], rot);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            for (int part = 0; part < 2; ++part) {
                const int from = part == 0 ? 0 : t_last + 1, to = part == 0 ? t_first : kBlock;
                if (to > from) {
                    s.z += lane >= from && lane < to ? coef : 0u;
                    if (wide) add_wide_terms(vb, tok, r, rot, from, to, s);
                    else add_terms<true>(vb, tok, r, rot, from, to, s);
                    dirty = true;
                }
                if (part == 0 && dirty) {
                    flush(sh, k, s, lane);
                    dirty = false;
                }
            }
            stretch = k + 1;
        } else if constexpr (SPLIT) {
            // The block's special tokens, and the pieces between them: the
            // first piece joins the stretch.
            // Blocks with wide V shifts are summed here too: giving the head up for them cost 51 us a step against 19
            // at batch 2, 464 tokens, Student-t(3) inputs (chunked kernel: 23).
            const bool special = (word & (kInit | kRescale)) != 0u;
            uint64_t m = __builtin_amdgcn_ballot_w64(special);
            const int count = __builtin_popcountll(m);
            uint32_t first = 0;
            if (lane == 0) first = atomicAdd(&sh.specials, static_cast<uint32_t>(count));
            first = uniform(first);
            if (first + count > static_cast<uint32_t>(kSpecials)) {
                if (lane == 0) sh.failed = 1u;
            } else {
                if (lane == 0) {
                    sh.hot_first[k] = first;
                    sh.hot_count[k] = static_cast<uint32_t>(count);
                }
                int e = k;
                for (int from = 0;;) {
                    const int t = m != 0u ? __builtin_ctzll(m) : kBlock;
                    if (t > from) {
                        s.z += lane >= from && lane < t ? coef : 0u;
                        if (wide) add_wide_terms(vb, tok, r, rot, from, t, s);
                        else add_terms<true>(vb, tok, r, rot, from, t, s);
                        dirty = true;
                    }
                    if (dirty) flush(sh, e, s, lane);
                    dirty = false;
                    if (m == 0u) break;
                    const uint32_t idx = first + static_cast<uint32_t>(count - __builtin_popcountll(m));
#pragma unroll
                    for (int i = 0; i < kRows; ++i)
                        if (i == t >> 3 && r == (t & 7)) *reinterpret_cast<v4i*>(&sh.code[idx][16 * c]) = vb.v[i];
                    if (lane == t) {
                        sh.sp_word[idx] = word;
                        sh.sp_exps[idx] = tok[lane].y;
                    }
                    e = kPool - 1 - static_cast<int>(idx);
                    from = t + 1;
                    m &= m - 1ull;
                }
            }
            if (dirty) flush(sh, k, s, lane);
            dirty = false;
            stretch = k + 1;
        }
    }
        const bool here = it + 1 < own_blocks;
        load_v(here ? pg : next, here ? begin + (wave + (it + 1) * kWaves) * kBlock : wave * kBlock,
               here || next_past == 0, vb);
    }
    if (dirty) flush(sh, stretch, s, lane);
    __syncthreads();
    const bool usable = uniform(sh.failed) == 0u;
    const bool staged = uniform(sh.staged) <= static_cast<uint32_t>(kStageRows);

    // The fold: the stretches' sums and the hot blocks in token order, one
    // thread per channel for Y, one wave for Z.
    const int g = (d >> 5) & 3;
    int32_t y = 0;
    uint32_t z = 0;
    const int32_t new_v = dequant_raw(sh.new_code[d & (kHeadDim - 1)], exps_shift(sh.new_exps, g));
    auto fold = [&](auto z_column) {
        // Stretch k, then hot block k's span, often one token; what block k + 1
        // needs is read ahead.
        constexpr bool Z = decltype(z_column)::value;
        const int col = stage_column(d);
        const uint4 table = sh.hot[lane];
        auto column = [&](uint32_t x, int k) {
            return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(x), k));
        };
        auto sum_of = [&](int k) { return Z ? static_cast<int32_t>(sh.pool_z[k]) : sh.pool[k][d]; };
        auto first_of = [&](int k) {
            const uint32_t row = min(column(table.y, k & 63), kStageRows - 1u);
            return Z ? sh.stage_z[row] : sh.stage[row][col];
        };
        int32_t sum = sum_of(0), first = first_of(0);
        float bound = Z ? 0.0f : sh.pool_b[0][g];
        for (int k = 0;; ++k) {
            const int32_t sum_k = sum, first_k = first;
            const float bound_k = bound;
            const int kn = min(k + 1, nbound);
            sum = sum_of(kn);
            if (!Z) bound = sh.pool_b[kn][g];
            first = first_of(kn);
            if (!Z && __builtin_amdgcn_ballot_w64(!bounded(y, bound_k)) != 0) {
                if (lane == 0) sh.unbounded = 1u;
                break;
            }
            y += sum_k;
            if (k == nbound) break;
            const uint32_t span = column(table.x, k), at = column(table.y, k);
            const int rows = static_cast<int>(span >> 16) - static_cast<int>(span & 0xffffu);   // none at a cut
            if (rows == 0) continue;
            y = __builtin_elementwise_add_sat(mulq17_wrap(y, column(table.z, k)), first_k);
            if (rows > 1) y = run_staged<Z>(sh, at + 1u, rows - 1, col, lane, y);
        }
    };
    if (folds && staged) {
        if (wave < 2) fold(std::false_type());
        else if (wave == 2) fold(std::true_type());
    }
    if (wave == 2 && lane == 0) {
        sh.z = static_cast<uint32_t>(y);
        sh.new_word = pos == 0 ? kInit : coef_word(sh.new_score, top, sh.lut);
    }
    __syncthreads();
    uint32_t new_word = uniform(sh.new_word);

    // Where that does not serve, the ordered pass over the range.
    if (folds && (!staged || uniform(sh.unbounded) != 0u)) {
        for (bool pieces = uniform(sh.unbounded) == 0u;; pieces = false) {
            y = ordered_pass(page_of(b, h), (SharedPtr)&sh, cap, begin, stop - begin, pieces ? 1 : 0, nbound, 0);
            if (wave == 2 && lane == 0) sh.z = static_cast<uint32_t>(y);
            __syncthreads();
            if (!pieces || uniform(sh.unbounded) == 0u) break;
        }
    }
    z = sh.z;

    bool add_new = true;                           // or the new token is in the merged sums
    if (SPLIT && !whole) {
        // Publish the range's entries; a split that cannot only says so.  Its own
        // entries 0 and 1 stay in LDS (sums in staging rows 0 and 1, values in
        // row 2), in case it is the one that folds: in registers they end up in
        // scratch memory, and reading that waits for the words just published.
        if (wave < 2) {
            int entries = 1;
            auto put = [&](int e, uint32_t av, uint32_t zv, float bv) {
                publish(slot_sums(mine, e) + d, tag, av);
                if (d == 0) publish(slot_misc(mine, e), tag, zv);
                if ((d & 31) == 0) publish(slot_misc(mine, e) + 2 + g, tag, __float_as_uint(bv));
                if (e < 2) sh.stage[e][d] = static_cast<int32_t>(av);
                if (e < 2 && d == 0) sh.misc[2 + 6 * e] = zv;
                if (e < 2 && (d & 31) == 0) sh.misc[4 + 6 * e + g] = __float_as_uint(bv);
            };
            auto put_special = [&](int e, uint32_t word, int32_t v) {
                publish(slot_values(mine, e) + d, tag, static_cast<uint32_t>(v));
                if (d == 0) publish(slot_misc(mine, e) + 1, tag, word);
                if (e == 1) sh.stage[2][d] = v;
                if (e < 2 && d == 0) sh.misc[3 + 6 * e] = word;
            };
            if (folds) {
                put(0, static_cast<uint32_t>(y), z, 0.0f);
            } else if (usable && static_cast<int>(uniform(sh.specials)) + __builtin_popcountll(cuts & ~hot) + 1 +
                                        (owner ? 1 : 0) <= kExactEntries) {
                put(0, static_cast<uint32_t>(sh.pool[0][d]), sh.pool_z[0], sh.pool_b[0][g]);
                for (int k = 0; k < nbound; ++k) {
                    const uint32_t first = uniform(sh.hot_first[k]), count = uniform(sh.hot_count[k]);
                    if (count == 0u) {             // a cut: an ordinary token that adds nothing
                        put_special(entries, 0u, 0);
                        put(entries, static_cast<uint32_t>(sh.pool[k + 1][d]), sh.pool_z[k + 1], sh.pool_b[k + 1][g]);
                        ++entries;
                    }
                    for (uint32_t i = 0; i < count; ++i) {
                        const int idx = static_cast<int>(first + i), e = kPool - 1 - idx;
                        uint32_t av = static_cast<uint32_t>(sh.pool[e][d]), zv = sh.pool_z[e];
                        float bv = sh.pool_b[e][g];
                        if (i + 1 == count) {
                            av += static_cast<uint32_t>(sh.pool[k + 1][d]);
                            zv += sh.pool_z[k + 1];
                            bv += sh.pool_b[k + 1][g];
                        }
                        put_special(entries, sh.sp_word[idx],
                                    dequant_raw(sh.code[idx][d], exps_shift(sh.sp_exps[idx], g)));
                        put(entries, av, zv, bv);
                        ++entries;
                    }
                }
                if (owner) {
                    put_special(entries, new_word, new_v);
                    put(entries, 0u, 0u, 0.0f);
                    ++entries;
                }
            } else {
                entries = static_cast<int>(kSlotFailed);
            }
            if (d == 0) {
                publish(mine + kSlotCount, tag, static_cast<uint32_t>(entries));
                sh.misc[1] = static_cast<uint32_t>(entries);
            }
        }
        // The count goes out from a wave that publishes nothing.
        constexpr unsigned kCountThread = kHeadDim;
        if (threadIdx.x == kCountThread) {
            const uint64_t n = __hip_atomic_fetch_add(arrival, uint64_t(1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sh.last = static_cast<uint32_t>(n) == static_cast<uint32_t>(nsplit - 1);
        }
        __syncthreads();
        if (!uniform(sh.last)) return;

        // The last split of the head to arrive folds the entries of all of
        // them.  Every split has counted, so its words land by themselves.
        // Entries 0 and 1 of every split come in one round of loads.  A wave
        // stops at the first split whose sums cannot be used; pool holds Y, and
        // pool_z Z, before each split.
        if (wave < 2) {
            bool ok = true;
            uint32_t budget = tail.merge_polls;
            constexpr int kMisc = 14;              // the maximum, the count and the words of entries 0 and 1
            const uint64_t own_tag = static_cast<uint64_t>(want) << 32;
            const uint64_t own_m = own_tag | sh.misc[min(lane, kMisc - 1)];
            const uint64_t own_a0 = own_tag | static_cast<uint32_t>(sh.stage[0][d]);
            const uint64_t own_a1 = own_tag | static_cast<uint32_t>(sh.stage[1][d]);
            const uint64_t own_v1 = own_tag | static_cast<uint32_t>(sh.stage[2][d]);
            uint64_t mw[kExactMaxSplits], a0[kExactMaxSplits], a1[kExactMaxSplits], v1[kExactMaxSplits];
            for (;;) {
#pragma unroll
                for (int j = 0; j < kExactMaxSplits; ++j) {
                    mw[j] = own_m;
                    a0[j] = own_a0;
                    a1[j] = own_a1;
                    v1[j] = own_v1;
                    if (j < nsplit && j != split) {
                        uint64_t* const p = slots + j * kExactSlotWords;
                        mw[j] = fetch(p + kSlotMax + min(lane, kMisc - 1));
                        a0[j] = fetch(slot_sums(p, 0) + d);
                        a1[j] = fetch(slot_sums(p, 1) + d);
                        v1[j] = fetch(slot_values(p, 1) + d);
                    }
                }
                bool stale = false;
#pragma unroll
                for (int j = 0; j < kExactMaxSplits; ++j) {
                    if (j < nsplit) {
                        const uint64_t count = __builtin_amdgcn_readlane(static_cast<int>(mw[j] >> 32), 1) ==
                                                       static_cast<int>(want)
                                                   ? static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(mw[j]), 1))
                                                   : 0u;
                        // of a failed split nothing but the maximum and the count is read
                        const bool failed = (count & kSlotFailed) != 0u, more = !failed && count > 1u;
                        stale |= count == 0u || (!failed && !current(a0[j], want)) ||
                                 (more && (!current(a1[j], want) || !current(v1[j], want))) ||
                                 ((lane == 0 || (!failed && lane >= 2 && lane < (more ? kMisc : 8) && lane != 3)) &&
                                  !current(mw[j], want));
                    }
                }
                if (__builtin_amdgcn_ballot_w64(stale) == 0) break;
                if (budget-- == 0u) {
                    ok = false;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            int fail_at = ok ? nsplit : 0;
            int32_t max_before = INT32_MIN;
            y = 0;
            z = 0u;
            sh.pool[0][d] = 0;
            if (lane == 0) {
                sh.pool_z[0] = 0u;
                sh.max_before[0] = INT32_MIN;
            }
#pragma unroll
            for (int j = 0; j < kExactMaxSplits; ++j) {
                if (j < nsplit && ok) {
                    if (j > 0) {
                        sh.pool[j][d] = y;
                        if (lane == 0) {               // the same values from both waves
                            sh.pool_z[j] = z;
                            sh.max_before[j] = max_before;
                        }
                    }
                    auto misc = [&](int i) -> uint32_t {
                        return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(mw[j]), i));
                    };
                    const uint32_t n = misc(1);
                    max_before = max(max_before, static_cast<int32_t>(misc(0)));
                    auto add = [&](uint32_t sum, uint32_t coefs, uint32_t bound_lo, uint32_t bound_hi) {
                        const float bv = __uint_as_float((d & 32) ? bound_hi : bound_lo);
                        ok = ok && __builtin_amdgcn_ballot_w64(!bounded(y, bv)) == 0;
                        y = static_cast<int32_t>(static_cast<uint32_t>(y) + sum);
                        z = (z + coefs) & kMask30;
                    };
                    if (n & kSlotFailed) {
                        ok = false;
                    } else {
                        add(static_cast<uint32_t>(a0[j]), misc(2), wave ? misc(6) : misc(4), wave ? misc(7) : misc(5));
                        if (n > 1) {
                            y = y_step(y, misc(9), static_cast<int32_t>(static_cast<uint32_t>(v1[j])));
                            z = z_step(z, misc(9));
                            add(static_cast<uint32_t>(a1[j]), misc(8), wave ? misc(12) : misc(10),
                                wave ? misc(13) : misc(11));
                        }
                        for (uint32_t e = 2; ok && e < n; ++e) {
                            uint64_t* const p = slots + j * kExactSlotWords;
                            uint64_t m, sum, v;
                            for (;;) {
                                m = fetch(slot_misc(p, static_cast<int>(e)) + min(lane, 5));
                                sum = fetch(slot_sums(p, static_cast<int>(e)) + d);
                                v = fetch(slot_values(p, static_cast<int>(e)) + d);
                                const bool stale = !current(m, want) || !current(sum, want) || !current(v, want);
                                if (__builtin_amdgcn_ballot_w64(stale) == 0) break;
                                if (budget-- == 0u) {
                                    ok = false;
                                    break;
                                }
                                __builtin_amdgcn_s_sleep(1);
                            }
                            auto extra = [&](int i) -> uint32_t {
                                return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(m), i));
                            };
                            y = y_step(y, extra(1), static_cast<int32_t>(static_cast<uint32_t>(v)));
                            z = z_step(z, extra(1));
                            add(static_cast<uint32_t>(sum), extra(0), wave ? extra(4) : extra(2),
                                wave ? extra(5) : extra(3));
                        }
                    }
                    if (!ok) fail_at = j;
                }
            }
            if (lane == 0) sh.fail_at[wave] = static_cast<uint32_t>(fail_at);
        }
        __syncthreads();
        const int fail_at = static_cast<int>(min(uniform(sh.fail_at[0]), uniform(sh.fail_at[1])));
        add_new = fail_at < nsplit;
        if (add_new) {
            const int32_t before = wave == 2 ? static_cast<int32_t>(sh.pool_z[fail_at])
                                             : sh.pool[fail_at][d & (kHeadDim - 1)];
            auto limbs = [&](int k) { return v4i{ql.w[k][0], ql.w[k][1], ql.w[k][2], ql.w[k][3]}; };
            y = run_rest(page_of(b, h), (SharedPtr)&sh, cap, fail_at * C, pos, sh.max_before[fail_at], limbs(0),
                         limbs(1), limbs(2), q3 ? 1 : 0, before);
            if (wave == 2 && lane == 0) sh.z = static_cast<uint32_t>(y);
            __syncthreads();
            z = sh.z;
            new_word = uniform(sh.new_word);
        }
    }
    if (add_new) {
        if (wave < 2) y = y_step(y, new_word, new_v);
        z = z_step(z, new_word);
    }

    // Y * 1/Z with the 18-bit quotient floor((2^34 + Z/2) / Z) (cpp:271-300),
    // RNE and a 32-bit wrap (cpp:1666-1710), and the integer-path A14/E8M0
    // (cpp:1694-1771, 2656-2682): group max of |raw| (INT32_MIN counts as
    // INT32_MAX), one float conversion, frexp exponent e, q =
    // trunc(clamp(raw*2^-17 * 2^(13-e) +- 0.5, +-8191)), code = e + 127.
    const size_t grp0 = static_cast<size_t>(b) * (kHeads * kGroupsPerHead) + h * kGroupsPerHead;
    if (wave < 2) {
        const uint32_t inv = z ? static_cast<uint32_t>(((1ull << 34) + (z >> 1)) / z) & 0x3ffffu : 0x3ffffu;
        const int32_t o = mulq17_wrap(y, inv);
        tail.out[static_cast<size_t>(b) * kModelDim + h * kHeadDim + d] = o;
        int32_t m = o == INT32_MIN ? INT32_MAX : (o < 0 ? -o : o);
#pragma unroll
        for (int s = 1; s < 32; s <<= 1) m = max(m, __shfl_xor(m, s));
        const float mx = static_cast<float>(m) * 0x1p-17f;
        int16_t q14 = 0;
        uint8_t code = 0;
        if (mx != 0.0f) {
            int e = 0;
            (void)frexpf(mx, &e);
            const float x = __fmul_rn(static_cast<float>(o) * 0x1p-17f, ldexpf(1.0f, 13 - e));
            float rr = x >= 0.0f ? __fadd_rn(x, 0.5f) : __fsub_rn(x, 0.5f);
            rr = fminf(fmaxf(rr, -8191.0f), 8191.0f);
            q14 = static_cast<int16_t>(static_cast<int>(rr));
            code = static_cast<uint8_t>(e + 127);
        }
        sh.q14[d] = q14;
        if (tail.act_scale != nullptr && (d & 31) == 0) tail.act_scale[grp0 + (d >> 5)] = code;
    }
    __syncthreads();
    if (tail.act_q != nullptr && d < kGroupsPerHead * 14) {
        const int gi = d / 14, w = d % 14;
        uint32_t word = 0;
        const int bit0 = 32 * w;
        for (int i = bit0 / 14; i <= (bit0 + 31) / 14 && i < 32; ++i) {
            const uint32_t val = static_cast<uint32_t>(static_cast<uint16_t>(sh.q14[gi * 32 + i])) & 0x3fffu;
            const int shl = 14 * i - bit0;
            word |= shl >= 0 ? (val << shl) : (val >> -shl);
        }
        reinterpret_cast<uint32_t*>(tail.act_q + (grp0 + gi) * 56)[w] = word;
    }
    if (SPLIT && !whole) {
        // Every split's words have been read: advance the generation (and
        // clear all of the head's slots when the tags wrap, those of splits
        // that only longer launches have among them, so that no word left from
        // 2^32-1 launches ago can pass for a current one).
        if (tag == 0xffffffffu)
            for (int i = d; i < exact_row_slots(b) * kExactSlotWords; i += kThreads)
                __hip_atomic_store(slots + i, uint64_t(0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (d == 0)
            __hip_atomic_store(arrival, static_cast<uint64_t>(tag == 0xffffffffu ? 0u : tag) << 32, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!more) break;
    // Nothing of this head is read from LDS any more but q14, which the next
    // one writes behind further barriers.
    h = next_h;
    b = next_b;
    pos = next_pos;
    pg.rsrc = next.rsrc;
    }
}

}  // namespace

hipError_t launch_exact(const StepArgs& a, int grid_splits, int cus, bool q17, hipStream_t s) {
    if (a.split_tokens <= 0 || a.split_tokens % kSplitQuantum != 0 || a.split_tokens > kExactMaxTokens ||
        a.kv.seq_cap > kMaxSeq || a.kv.layers > 0xffff || a.batch < 1 || a.batch > kMaxBatchPerLaunch || cus < 1 ||
        grid_splits < 1 || (grid_splits > 1 && grid_splits > exact_splits(a.batch)))
        return hipErrorInvalidValue;
    StepPreload p = step_preload(a);
    // Unsplit launches: one workgroup per CU (LDS holds no second one) takes
    // heads in turn, back and forth over the rows (longest first), so that a
    // ragged batch ends evenly.
    const int rows = std::min({a.batch, std::max(cus / kHeads, 1), 255});   // of 32 workgroups
    if (grid_splits == 1)
        p.dispatch = (p.dispatch & StepPreload::kRowsListed) | static_cast<uint32_t>(a.batch - 1) << 16 |
                     static_cast<uint32_t>(rows) << 24;
    const dim3 grid = grid_splits > 1 ? dim3(grid_splits, kHeads, a.batch) : dim3(rows * kHeads);
    const void* workspace = a.partials;
#define SKV_EXACT(Q17, SPLIT)                                                                                        \
    exact_kernel<Q17, SPLIT><<<grid, kThreads, 0, s>>>(p.layer_pages, p.geometry, p.dispatch, a.q, a.k, a.v, a.lut, \
                                                       workspace, a)
    if (grid_splits > 1) {
        if (q17) SKV_EXACT(true, true);
        else SKV_EXACT(false, true);
    } else {
        if (q17) SKV_EXACT(true, false);
        else SKV_EXACT(false, false);
    }
#undef SKV_EXACT
    return hipGetLastError();
}

}  // namespace swiftkv
