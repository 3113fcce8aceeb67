// rules.hpp -- which kernel of a family a call takes, where that follows from
// its sizes and addresses alone: code without HIP, so that the choices can be
// checked on any machine. What each line rests on stands beside it.
#pragma once

#include <cstdint>

#include "../../include/vkml_hip.h"

namespace vkml::rules {

// ---------------------------------------------------------------- vkml_matmul

// How k_matmul (k_matmul_f32.hip) loads its operands: element by element; b
// four at a time; a and b four at a time (rows of whole, aligned vec4s, and a
// tile's offsets from its own base in 32 bits).
enum Loads { kScalar = 0, kVecB = 1, kVecAB = 2 };

// The loads of a product with a float b: a's vec4s lie along k, b's along k
// if it is transposed and along n otherwise. The offsets of a tile, up to 128
// rows of a or b, from its base fit 32 bits, whatever a and b hold in all.
inline Loads float_loads(const vkml_matmul_params& p, uintptr_t a, uintptr_t b) {
    const uint32_t len = p.b_transposed ? p.k : p.n;
    const bool vec_a = p.k % 4 == 0 && a % 16 == 0 && p.k < (1u << 25) && len < (1u << 25);
    const bool vec_b = len % 4 == 0 && p.b_stride % 4 == 0 && b % (p.b_type == VKML_F32 ? 16 : 8) == 0;
    if (vec_b && vec_a) return kVecAB;
    return vec_b && !p.b_transposed ? kVecB : kScalar;
}

// A quantized b's codes come four at a time whatever their address; a's
// loads follow a's alignment (k is whole blocks).
inline Loads quant_loads(const vkml_matmul_params& p, uintptr_t a) { return a % 16 == 0 && p.k < (1u << 25) ? kVecAB : kScalar; }

// A wave's tile of the product: 16 nc rows by 16 r columns.
struct WaveTile {
    int r, nc;
};

// The larger a tile, the fewer operands it stages; the smaller, the more
// waves and the less padding. The lines are at the waves with work that a
// tile gives: of masked scores the part of the keys that the average query
// sees (of probs v a mask shortens the sums and leaves every tile). Measured (us; wave tiles of 32 x 64, 32 x 32, 16 x 32 and 16 x 16):
// scores of 2048 queries by 4096 keys, 32 heads of 128, 996, 1015, 1107, 1249;
// 8192 x 8192 x 128 295, 298, 329, 376; 2048 x 8192 x 2048 1111, 1095, 1155,
// 1275; probs v at those 2048 queries 952, 909, 942, 1014; 900 x 8192 x 2048
// 603, 576, 556, 588; 200 x 14336 x 4096 626, 587, 533, 499; 131 x 2048 x
// 8192 886, 471, 283, 218. Every tile of columns widens a quantized b again,
// so the taller tiles win from fewer waves on: q4_K 512 x 8192 x 2048 387,
// 335, 350, 401; 512 x 4096 x 4096 611, 383, 387, 418; 1000 x 2048 x 2048 309,
// 193, 195, 211; 300 x 8192 x 2048 383, 270, 234, 259; 131 x 8192 x 2048 297,
// 190, 158, 146; q4_0 2048 x 14336 x 4096 3846, 3924, -, -. The q4_K 32 x 64
// tile, whose headers take the registers that its loads would be in flight in,
// loses everywhere (2048 x 14336 x 4096 4244 against 4109).
inline WaveTile wave_tile(const vkml_matmul_params& p) {
    const double seen = p.causal && p.b_transposed ? (p.causal_offset + 0.5 * p.m) / (p.causal_offset + 1.0 * p.m) : 1.0;
    const auto waves = [&](uint64_t r, uint64_t nc) {
        return seen * static_cast<double>((p.m + 16 * nc - 1) / (16 * nc) * ((p.n + 16 * r - 1) / (16 * r)) * p.batches);
    };
    if (p.b_type >= VKML_Q8_0) {
        if (p.b_type != VKML_Q4_K && waves(4, 2) >= 16384) return {4, 2};
        if (waves(2, 2) >= 3072) return {2, 2};
        if (waves(2, 1) >= 3584) return {2, 1};
        return {1, 1};
    }
    // The smallest tile multiplies whole chunks of 64 k's, the others chunks of
    // 32 or parts of one: short sums that leave half of a last 64 empty go to
    // the others from fewer waves on (f16, 130 x 9532 x 72 12.0, 10.5, 8.7, 12.1;
    // 1188 x 2272 x 88 18.9, 15.6, 16.4, 19.9; 518 x 5040 x 16 7.7, 6.6, 6.5,
    // 12.9, where the kernel before took 7.9).
    // Element loads (a ragged k) and b [k, n]'s tails, which only the 32 x 64
    // tile cuts, leave less of that.
    const bool half = (p.k - 1) % 64 < 32, tiny = half && p.k <= 32 && p.k % 4 == 0, brief = half && p.k <= 160 && (p.b_transposed || p.k <= 32);
    if (waves(4, 2) >= (tiny ? 4096 : 16384)) return {4, 2};
    if (waves(2, 2) >= (tiny ? 2048 : 8192)) return {2, 2};
    if (waves(2, 1) >= (tiny ? 512 : brief ? 1024 : 6144)) return {2, 1};
    return {1, 1};
}

// Whether a 32- or 16-row by 32 tile leaves out the last chunk's k's past the
// sums (chunks of 32 k's): short sums of a transposed float b that end in a
// chunk's first half, as the scores of heads of 80. It is a loop of other than
// constant length, which costs whole chunks (us without and with it, 32 x 32
// tiles: scores of 2048 queries by 4096 keys, 8 heads of 80, 180, 162; of 72
// 180, 162; of 128 229, 236; 900 x 8192 x 2048 570, 590; 2048 queries by 4096
// keys' probs v, 32 heads of 128 in 16 x 32 tiles, 907, 945). The 32 x 64 tile
// always does (an f32 b's probs v of 1000 queries by 2001 keys 334, 285: it
// spills fewer registers so; 8192 columns of 2048 k's within 2% either way),
// the 16 x 16 tile, a chain of chunks that it makes 4 to 10% longer, never.
inline bool cut_last_chunk(const vkml_matmul_params& p) {
    return p.b_transposed && p.b_type <= VKML_BF16 && p.k <= 256 && (p.k - 1) % 32 < 16;
}

// ---------------------------------------------------------------- vkml_matmul_dot

// A wave's tile in k_matmul_dot (k_matmul.hip): 16 rt rows by 16 ct columns;
// four of them side by side are a workgroup's.
struct DotTile {
    int rt, ct;
};

// Tiles of 64 x 128, 32 x 128, 16 x 128 and 16 x 64 outputs: a larger one
// stages less for each output and scales more of them at a time, a smaller one
// gives the SIMDs more waves, and the formats differ in the registers that
// their scales take. The lines, by waves of a 64 x 32 or 32 x 32 tile (1024
// SIMDs), are where the times cross over. Measured (us; those four):
// q4_K: 512 x 2048 x 2048 (1024 waves) 36, 22, 17.9, 19.4; 384 x 4096 x 4096
// (1536) 68, 50, 42.6, 53; 800 x 2048 x 8192 (1600) 134, 93.4, 114, 114; 512 x
// 14336 x 4096 158, 134, 173, 215; 1000 x 14336 x 4096 264, 258, 336, 411; 4096
// x 4096 x 4096 287, 292, 383, 469; 40 and 64 x 14336 x 4096 (896) 29.1 and
// 36.2 in 16 x 64, 31.9 and 33.2 in 16 x 128.
// q4_0: 256 x 4096 x 4096 (1024) 69, 43, 37, 31; 300 x 4096 x 4096 (1280) 69,
// 50, 48, 36; 160 x 9216 x 4096 (1440) 70, 50, 47.8, 49.5; 512 x 4096 x 4096
// (2048) 71, 52, 57, 58.
// q8_0: 256 x 4096 x 4096 68, 41, 36, 34; 131 x 8192 x 2048 (1280) 36, 25.4,
// 26.9, 26.5; 128 x 14336 x 4096 72, 51, 75, 63; 4096 x 4096 x 4096 334, 307,
// 449, 448; with f32 scales 131 x 8192 x 2048 32, 24.3, 24.3, 21.5.
// q4_1: 352 x 4096 x 4096 (1408) 84, 52.7, 48.2, 49.7; 265 x 5574 x 1056 (1575)
// 24, 17.3, 16.1, 18.7; 4096 x 4096 x 4096 311, 299, 433, 453; with f32 scales 384 x 4096 x
// 4096 77, 56, 48, 53; 3000 x 6144 x 4096 422, 386, 456, 567.
// (16 x 256 and 32 x 256 tiles lost throughout: 213 to 241 VGPRs. A second
// chunk in flight in registers gained up to 4% at q4_K products of few
// workgroups and lost 15 to 20% on the other formats, whose scales take more
// registers.)
constexpr bool dot_has_64_rows(uint32_t b_type) { return b_type == VKML_Q4_0 || b_type == VKML_Q4_K; }
// From how many waves of a 32 x 32 tile on a 16 x 128 one (not q8_0).
constexpr uint64_t dot_16x128_line(uint32_t b_type, bool f16_scales) {
    return b_type == VKML_Q4_0 ? 1400 : b_type == VKML_Q4_1 && f16_scales ? 1280 : b_type == VKML_Q8_0 ? ~0ull : 900;
}

inline DotTile dot_tile(uint32_t b_type, bool f16_scales, uint32_t m, uint32_t n) {
    const auto waves = [&](uint64_t rt, uint64_t ct) { return ((m + 16 * rt - 1) / (16 * rt)) * ((n + 16 * ct - 1) / (16 * ct)); };
    if (dot_has_64_rows(b_type) && waves(4, 2) >= 8192) return {4, 2};
    // (q4_0's and q4_1's 16 x 128 tile holds three workgroups a compute unit;
    // one more round of them loses: q4_1 909 x 1737 x 4096, 798 workgroups,
    // 52.8, 71.5 us, 909 x 1664 x 4096, 741, 52.2, 49.2)
    const bool mid = waves(2, 2) >= dot_16x128_line(b_type, f16_scales);
    const bool second_round = b_type != VKML_Q4_K && waves(1, 2) > 4 * 3 * 256;
    if (waves(2, 2) >= (b_type == VKML_Q8_0 && f16_scales ? 1280 : 1600) || (mid && second_round)) return {2, 2};
    if (mid) return {1, 2};
    return {1, 1};
}

// How k_matmul_dot's rows x columns tiles lie on its grid. Workgroups go to the
// eight XCDs in turn, each with an L2 of its own. With whole eights of column
// tiles, a grid (columns, rows) leaves each XCD an eighth of them, whose
// weights its row tiles find in its L2. With any other number every XCD reads
// all of the weights, from the last-level cache: q8_0 1719 x 9223 x 6848 (73
// columns of 32 x 128 tiles) took 790 us where 72 columns took 508. Then the
// tiles are numbered band by band of an eighth of the columns, row by row in a
// band, and each XCD takes a contiguous eighth of that order (width 0: the
// plain grid): 524 us; 2000 x 9000 x 8192 884 -> 688, q4_0 1719 x 9223 x 4160
// 361 -> 281.
#ifdef __HIPCC__
#define VKML_RULES_BOTH __host__ __device__
#else
#define VKML_RULES_BOTH
#endif
struct DotBands {
    uint32_t rows, columns;
    uint32_t width;  // columns of a band
    uint32_t share;  // tiles of an XCD

    // The tile of workgroup i of 8 share; whether it has one.
    VKML_RULES_BOTH bool tile(uint32_t i, uint32_t& row, uint32_t& col) const {
        const uint32_t s = i % 8 * share + i / 8;
        if (s >= rows * columns) return false;
        const uint32_t band = s / (width * rows), at = s % (width * rows), first = band * width;
        const uint32_t w = columns - first < width ? columns - first : width;
        row = at / w;
        col = first + at % w;
        return true;
    }
};

// (A launch of few tiles reads little twice; a grid's work items along x, 256
// a tile, fit 32 bits.)
inline DotBands dot_bands(uint32_t rows, uint32_t columns) {
    const uint64_t tiles = static_cast<uint64_t>(rows) * columns;
    const bool bands = columns % 8 != 0 && columns > 8 && rows >= 8 && tiles < (1u << 23);
    return {rows, columns, bands ? (columns + 7) / 8 : 0, static_cast<uint32_t>((tiles + 7) / 8)};
}

// The last chunk of K, 8 blocks of 32, in k_matmul_dot: whole
// (no masks, no branch); all its blocks, those past K as zeros; or only the
// groups of blocks (one, two or, in the 16 x 64 tile, four) that hold some,
// at a branch a group in every chunk.
enum DotTail { kWholeTail = 0, kMaskedTail = 1, kCutTail = 2 };

// rt, ct: a wave's tile, 16 rt rows by 16 ct columns. Measured (us; masked,
// cut): q8_0 300 x 4096 (32 x 128 tiles), K of 32 5.7, 4.4; 128 5.7, 5.0; 224
// 5.8, 5.7; 2080 equal. In the 16 x 64 tile the cut saves half a chunk or
// nothing, and its branch costs 5%: q8_0 64 x 4096, K of 32 3.1, 2.9; q4_1 64 x
// 4096, 224 3.13, 3.3, 2080 10.9, 11.3.
inline DotTail dot_tail(int rt, int ct, uint32_t k) {
    if (k % 256 == 0) return kWholeTail;
    return rt * ct > 1 || (k % 256 <= 128 && k <= 1024) ? kCutTail : kMaskedTail;
}

// ---------------------------------------------------------------- vkml_gemv_dot

// The rounds of 512 values that the kernel of 2 to 8 activation rows
// (k_gemv_dot_rows) stages at a time. Rows shorter than a chunk load and stage
// its other rounds for nothing. Measured (us; four rounds, two, one; the
// kernel before it, which staged nothing): q4_K, three rows, 30000 x 256 9.8,
// 6.7, 5.2 (6.0); q8_0, five rows, 30000 x 512 8.5, 6.8, 5.4 (6.4); the mean
// over the formats and 2 to 8 rows against that kernel at 30000 x 768 0.93,
// 1.19, 1.28 times as fast, 8192 x 1024 1.05, 1.23, 1.18, 2048 x 1536 1.17,
// 1.15, 1.15, 2048 x 2048 1.26, 1.25, 1.16.
inline uint32_t rows_chunk(uint32_t k) { return k <= 768 ? 1 : k <= 1024 ? 2 : 4; }

// ---------------------------------------------------------------- vkml_gemv

// Whether a float GEMV with rows of up to 256 values (k_gemv_float4) takes one
// row of b a half wave: with few outputs the launch is one wave's chain of
// loads, sums and tree, which more rows a lane lengthen; with many the loads
// in flight a lane matter. Measured as times as fast as the element-wise
// kernel (the mean over the float types and k of 4 to 128; one row a half
// wave, against four, or two from three rows of a on): one row of a, 1000
// outputs 1.10, 0.91, 8000 1.32, 1.24, 64000 1.96, 2.26; two, 1000 1.16,
// 0.86, 8000 1.32, 1.16, 64000 1.76, 1.82; three, 4000 1.18, 1.15, 8000 1.24,
// 1.29; five, 1000 1.16, 1.01, 4000 1.16, 1.12, 8000 1.17, 1.21, 64000 1.12,
// 1.37; eight, 1000 1.18, 1.04, 4000 1.19, 1.15, 9600 1.04, 1.17 (f32 rows of
// 192 and 256 values, 5000 outputs, eight: 4.7 us, 4.4).
inline bool gemv_row_each(uint32_t m, uint32_t n, uint32_t batches) { return static_cast<uint64_t>(n) * batches <= (m <= 2 ? 8192 : 4096); }

// Whether one row of a by an f32 b of long rows reads a from the caches
// (k_gemv_float4, eight steps at once) instead of staging it
// (k_gemv_float4_rows). A b past the 256 MiB of the last-level cache comes
// from memory at its rate, and the staging's barriers cost more than its reads
// save. Measured (us; cached, staged; the element-wise kernel): 12000 x 8192
// 69.2, 73.6 (68.9); 16000 x 8192 90.6, 93.3 (88.9); 32000 x 4096 84.7, 85.7
// (89.6); up to that size 8192 x 8192 52.2, 50.6 (54.2); 32000 x 2048 43.9,
// 42.8 (46.6).
inline bool gemv_row_cached(const vkml_gemv_params& p) {
    return p.b_type == VKML_F32 && p.m == 1 && p.k >= 4096 && static_cast<uint64_t>(p.n) * p.k > (1u << 26);
}

// ---------------------------------------------------------------- vkml_attend_prompt_fast

// Whether k_attend_prompt_fast's blocks are of 64 keys instead of 32: half the
// waits, barriers and maxima a key and twice the independent matrix
// instructions between them, against up to half a block of masked keys more,
// where the keys are few and an odd number of 32s, and, at head_dim 128, LDS
// that leaves two workgroups a compute unit instead of four. A third round of
// those pays only where the tiles' lengths differ (the longest start first),
// as they do from position 0. Measured (us; 32, 64; 32 heads on 8 KV heads):
// head_dim 128, 9 queries 4.3, 4.9; 40 5.6, 5.8; 64 6.4, 6.0; 90 7.5, 7.8; 128 8.8, 7.9; 150
// 9.9, 9.7; 192 11.0, 9.9; 300 15.6, 13.7; 64 after 1000 keys 42.2, 34.6; 1000
// after 37 43.1, 38.3; 1100 (552 workgroups) 46.2, 39.7, after 4000 keys 236,
// 273; 1500 (752) 61.6, 53.3; 2048 (1024) 88.6, 93.2; head_dim 64, 9 queries
// 3.4, 3.8; 64 4.56, 4.33; 90 5.36, 5.48; 128 6.2, 5.5; 1000 28.8, 23.1; 2048
// after 2048 keys 151, 142.
inline bool wide_blocks(const vkml_attend_prompt_params& p, uint32_t workgroups, uint32_t compute_units) {
    const uint32_t keys = p.first + p.t;
    if (keys <= 48 || (keys <= 128 && (keys + 31) / 32 % 2 != 0)) return false;
    return p.head_dim == 64 || workgroups <= 2 * compute_units || (workgroups <= 3 * compute_units && p.first < p.t);
}

}  // namespace vkml::rules
