// k_matmul.hip -- the int8 matrix product for many rows (prefill): the
// reference's shaders/matmul_dot.comp (src/ops/matmul.cpp:246-259), c = a b^T
// with a [M, K] Q8_0 activations (f32 scales) and b [N, K] quantized weights,
// on gfx950's matrix cores.
//
// Order (matmul_dot.comp:134-160). Each output is a sum over K's 32-value
// blocks in order: the block's exact integer dot product of the two codes,
// scaled in f32 and added to the output's accumulator,
//   q8_0 / q4_0: acc += float(sum) * (sa * sb)
//   q4_1 / q4_K: acc += sa * (float(sum) * sb + float(asum) * ob)
// (asum: the block's sum of a's codes; q4_K as its q4_1 form, scale
// f16(d sc) and offset f16(-dmin m) per 32 values, src/io/gguf.cpp:603-617).
// One v_mfma_i32_16x16x32_i8 computes the integer sums of one block for a
// 16 x 16 tile of outputs exactly, so the matrix cores do the dot products
// and the VALU applies the scales per block, in the reference's order.
//
// Mapping. A workgroup of four waves computes a tile of c, each wave 16 RT
// rows by 16 CT columns (RT x CT matrix instructions a block; 64 x 32 for
// large products, smaller tiles for short prompts so every SIMD gets work).
// Lane l of a wave holds, for a 16 x 16 instruction, a's row l % 16 and b's
// column l % 16 at the block's values 8 (l / 16) .. 8 (l / 16) + 7 (one
// 8-byte operand each), and gets the results for rows 4 (l / 16) .. + 3 of
// column l % 16. K runs in chunks of 8 blocks, staged in LDS with 16-byte
// loads a chunk ahead in registers: the operands, every row's
// (scale, code sum) and every column's (scale, offset) per block; the
// scaling reads four rows' values as one 16-byte word.
//
// What bounds it. The scaling costs 4 operations per output and block (the
// offset formats' six folded into four, as kSumBiasBits says), which issue at
// about 1.04 ns a wave64 instruction on a SIMD with waves enough, and the int8
// matrix instructions, 6.8 ns each, run beside them only in part. One operation
// in four is an outer product of a row tile's and a column tile's values, which
// the matrix unit forms for sixteen outputs a lane at once, 0.85 ns each
// (add_tiles): 22.7 ns for a lane's four outputs of a block, 740 TOP/s, when
// nothing waits and nothing overlaps. The large products reach 480 TOP/s, the
// 512-row ones 360 to 440: they fill 57 to 80% of their time. Against kernels
// that formed that product on the VALU, and loaded the operands of small
// products from memory block by block (us): 512 x 14336 x 4096 (q4_K) 152 ->
// 141, 512 x 4096 x 14336 179 -> 164, 1000 x 8192 x 3072 (q4_1) 140 -> 121; 131
// x 2048 x 8192 (q8_0) 116 -> 39, 37 x 4096 x 14336 135 -> 63, 9 x 4096 x 4096
// 33.5 -> 19.8.
#include <algorithm>

#include "../../include/vkml_hip.h"
#include "device.hpp"
#include "internal.hpp"
#include "rules.hpp"

using namespace vkml::dev;
using namespace vkml::rules;

namespace {

constexpr uint32_t kT = 256;      // four waves
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

struct MatmulDotArgs {
    const uint8_t* a;     // [M, K] activation codes
    const float* a_scales;  // [M, K / 32]
    const uint8_t* b;     // weight codes (layout per format)
    const void* b_scales;  // per-block scales (q4_K: the 16-byte super-block headers)
    float* out;           // [M, N]
    uint32_t m, n, k;
    const float* residual;  // [M, N] added to each output, or null
    DotBands bands;  // the order of the tiles over the grid
};

// out[row, col] = v, or residual[row, col] + v (the binary add that
// follows the o and down projections, the same f32 sum).
__device__ __forceinline__ void store_out(const MatmulDotArgs& p, uint32_t row, uint32_t col, float v) {
    const uint64_t at = static_cast<uint64_t>(row) * p.n + col;
    p.out[at] = p.residual ? p.residual[at] + v : v;
}

__device__ __forceinline__ float f16_at(const void* p, uint64_t i) { return f16_bits_to_float(ldg(static_cast<const uint16_t*>(p) + i)); }

// Four Q4_0 values as signed bytes, the low (shift 0) or high (shift 4)
// nibbles of a word minus 8 (matmul_dot.comp:71-73).
__device__ __forceinline__ uint32_t q4_signed(uint32_t word, uint32_t shift) {
    return (((word >> shift) & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u;
}

// Column n's scale and offset for block blk (q8_0 / q4_0: offset unused).
template <int FMT, bool F16S>
__device__ __forceinline__ void b_block_scale(const MatmulDotArgs& p, uint32_t n, uint32_t blk, float& s, float& o) {
    const uint64_t block = static_cast<uint64_t>(n) * (p.k / 32) + blk;
    o = 0.0f;
    if constexpr (FMT == VKML_Q8_0 || FMT == VKML_Q4_0) {
        s = F16S ? f16_at(p.b_scales, block) : ldg(static_cast<const float*>(p.b_scales) + block);
    } else if constexpr (F16S) {
        const uint32_t so = ldg(static_cast<const uint32_t*>(p.b_scales) + block);  // f16 scale | f16 offset << 16
        s = f16_bits_to_float(so & 0xFFFFu);
        o = f16_bits_to_float(so >> 16);
    } else {
        const float2 so = ldg(static_cast<const float2*>(p.b_scales) + block);
        s = so.x;
        o = so.y;
    }
}

constexpr uint32_t kChunk = 8;  // blocks of K a chunk (a q4_K super-block)

// The offset formats with f16 scales (q4_K, q4_1 with f16 scales) take the
// reference's six scaling operations, cvt, mul, mul, add, mul, add, as
// four: fma, fma, mul, add, with every result bit for bit the same.
//  - The matrix instruction starts its accumulator at the int32 bits of the
//    f32 1.5 * 2^23, so each block sum comes out as the bits of the f32
//    1.5 * 2^23 + sum, exactly (|sum| <= 32 * 128 * 15 < 2^22). Then
//    fma(that, sb, -1.5 * 2^23 * sb) forms the exact sum * sb and rounds it
//    once: float(sum) * sb, with no conversion. -1.5 * 2^23 * sb is exact
//    because sb is an f16 value (11 significant bits, 13 after the 3).
//  - asum * ob is exact (|asum| <= 32 * 128 = 2^12 has at most 12
//    significant bits, ob is an f16 value, and the smallest nonzero
//    product, 2^-24, is a normal f32), so fma(asum, ob, x) rounds x +
//    asum * ob once, as the reference's add of the rounded product does.
// Signs of zero can differ in the intermediate (an exact zero sum is +0,
// not -0 * sb), but no accumulator starting at +0 ever sees the
// difference: +0 + -0 is +0, and a nonzero accumulator ignores both.
constexpr int32_t kSumBiasBits = 0x4B400000;  // the f32 1.5 * 2^23
constexpr float kSumBias = 12582912.0f;

template <int FMT, bool F16S>
constexpr bool kFoldScaling = FMT == VKML_Q4_K || (FMT == VKML_Q4_1 && F16S);

template <int FMT, bool F16S>
__device__ __forceinline__ v4i sum_start() {
    constexpr int32_t b = kFoldScaling<FMT, F16S> ? kSumBiasBits : 0;
    return v4i{b, b, b, b};
}

// A 16 RT x 64 CT tile with its operands staged in LDS: per 8-block chunk
// the workgroup copies the chunk's A rows (16 RT x 256 bytes) and B columns
// (64 CT x 128 bytes, 256 for q8_0) with 16-byte loads, a chunk ahead in
// registers, and the matrix instructions read their operands from LDS. Each staging thread's A bytes are whole blocks of one row (two at RT =
// 4, one below; at RT = 1 half the threads stage A), so it also sums their
// codes.
template <int FMT, bool F16S, int RT, int CT>
struct StagedChunk {
    static constexpr bool kOffset = FMT == VKML_Q4_1 || FMT == VKML_Q4_K;
    static constexpr uint32_t TM = 16 * RT, TN = 64 * CT;     // the tile
    static constexpr uint32_t kABlocks = RT >= 2 ? RT / 2 : 1;  // a staging thread's A blocks (of one row)
    static constexpr uint32_t kAThreads = TM * kChunk / kABlocks;  // threads that stage A
    static constexpr uint32_t kBBytes = FMT == VKML_Q8_0 ? 256 : 128;  // a column's bytes a chunk
    static constexpr uint32_t kAStride = 272, kBStride = kBBytes + 16;  // padded rows: no bank conflicts
    static constexpr uint32_t kBLoads = kBBytes * TN / 16 / kT;         // 16-byte B loads a thread
    static constexpr uint32_t kSThreads = 2 * TN < kT ? 2 * TN : kT;     // threads that stage columns' scales, four blocks of
    static constexpr uint32_t kSCols = 2 * TN / kSThreads;              // this many columns each
    uint4 a[2 * kABlocks];
    uint4 b[kBLoads];
    float sa[kABlocks];
    uint4 header[kSCols];
    float s[kSCols][4], o[kSCols][4];
};

template <int FMT, bool F16S, int RT, int CT>
struct StagedLds {
    using S = StagedChunk<FMT, F16S, RT, CT>;
    alignas(16) uint8_t a[S::TM * S::kAStride];
    alignas(16) uint8_t b[S::TN * S::kBStride];
    alignas(16) float sa[kChunk][S::TM];
    alignas(16) float asum[kChunk][S::kOffset ? S::TM : 4];
    float sb[kChunk][S::TN];
    float ob[kChunk][S::kOffset ? S::TN : 1];
};

// Keeps the VALU instructions before it before those after it; the others
// (LDS reads, matrix instructions, scalar ones) may cross.
__device__ __forceinline__ void valu_stage() { __builtin_amdgcn_sched_barrier(0x3FC); }

// One output's contribution of one block, sa (sum sb + asum ob) or
// sum (sa sb) (matmul_dot.comp:155-160), from the matrix instruction's
// result d (biased where the scaling folds; nsb = -1.5 * 2^23 * sb).
template <int FMT, bool F16S>
__device__ __forceinline__ float block_term(int32_t d, float sa, float asum, float sb, float nsb, float ob) {
#pragma clang fp contract(off)
    if constexpr (kFoldScaling<FMT, F16S>) {
        const float x = __builtin_fmaf(__builtin_bit_cast(float, d), sb, nsb);
        return sa * __builtin_fmaf(asum, ob, x);
    } else if constexpr (FMT == VKML_Q4_1 || FMT == VKML_Q4_K) {
        return sa * (static_cast<float>(d) * sb + asum * ob);
    } else {
        return static_cast<float>(d) * (sa * sb);
    }
}

// A block's operands of the scaling: the wave's rows' scales and code sums
// (rows 4 g .. + 3 of each row tile), its columns' scales and offsets.
template <int RT, int CT>
struct BlockStats {
    float4 sa[RT], asum[RT];
    float sb[CT], nsb[CT], ob[CT];
};

// The results of G blocks' RT x CT tiles (d) into the accumulators, block by
// block in each: one operation of all sixteen terms a lane, then the next, so
// that no operation waits for the one before it. (Left to itself the compiler
// forms each term's four dependent operations in a row.)
template <int FMT, bool F16S, int RT, int CT, int G>
__device__ __forceinline__ void add_tiles(const v4i (&d)[G][RT][CT], const BlockStats<RT, CT> (&st)[G], const StagedLds<FMT, F16S, RT, CT>& l,
                                          uint32_t block, uint32_t wave, uint32_t lane, float (&acc)[RT][CT][4]) {
#pragma clang fp contract(off)
    static_assert(RT * CT * G == 4);
    // What a row and a column give together, the code sums times the offsets
    // or the two scales, are outer products of a row tile's and a column
    // tile's sixteen: one v_mfma_f32_16x16x1_4b_f32 forms them for four tiles
    // from one value a lane of each, each rounded as the VALU rounds it
    // (fma(asum, ob, x) on the scaled sums; sa * sb on zeros, where a -0 comes
    // out +0, which no accumulator can tell).
    constexpr bool kScales = FMT == VKML_Q8_0 || FMT == VKML_Q4_0;
    if constexpr (kFoldScaling<FMT, F16S> || kScales) {
        const uint32_t blk = lane / 16, li = lane % 16, q = blk / (RT * CT), cl = 16 * CT * wave + 16 * (blk / RT % CT) + li;
        float row, col;
        if constexpr (kScales) {
            row = l.sa[block + q][16 * (blk % RT) + li];
            col = l.sb[block + q][cl];
        } else {
            row = l.asum[block + q][16 * (blk % RT) + li];
            col = l.ob[block + q][cl];
        }
        v16f t;
        valu_stage();
        if constexpr (kScales) {
            const v16f u = __builtin_amdgcn_mfma_f32_16x16x1f32(row, col, v16f{}, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 16; ++j) t[j] = static_cast<float>(d[j / (4 * RT * CT)][j / 4 % RT][j / (4 * RT) % CT][j % 4]);
            valu_stage();
#pragma unroll
            for (int j = 0; j < 16; ++j) t[j] = t[j] * u[j];
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int b = j / (4 * RT * CT), r = j / 4 % RT, c = j / (4 * RT) % CT;
                const int sum = d[b][r][c][j % 4];  // (bit_cast of a vector's element itself takes element 0)
                t[j] = __builtin_fmaf(__builtin_bit_cast(float, sum), st[b].sb[c], st[b].nsb[c]);
            }
            t = __builtin_amdgcn_mfma_f32_16x16x1f32(row, col, t, 0, 0, 0);
            valu_stage();
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int b = j / (4 * RT * CT), r = j / 4 % RT, i = j % 4;
                const float4 s4 = st[b].sa[r];
                t[j] = (i == 0 ? s4.x : i == 1 ? s4.y : i == 2 ? s4.z : s4.w) * t[j];
            }
        }
        valu_stage();
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j / 4 % RT][j / (4 * RT) % CT][j % 4] += t[j];
        valu_stage();
    } else {
        // q4_1 with f32 scales: the reference's operations.
#pragma unroll
        for (int b = 0; b < G; ++b)
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const float sa[4] = {st[b].sa[r].x, st[b].sa[r].y, st[b].sa[r].z, st[b].sa[r].w};
                const float asum[4] = {st[b].asum[r].x, st[b].asum[r].y, st[b].asum[r].z, st[b].asum[r].w};
#pragma unroll
                for (int c = 0; c < CT; ++c)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc[r][c][i] += block_term<FMT, F16S>(d[b][r][c][i], sa[i], asum[i], st[b].sb[c], st[b].nsb[c], st[b].ob[c]);
            }
    }
}

// The same for the 64 x 32 wave tile, one block: a row tile's terms as the
// compiler orders them (its chains overlap those of the next row tile's, and
// sixteen at a time needed registers that cost a wave: 4096 x 14336 x 4096
// 1079 against 1010 us).
template <int FMT, bool F16S, int RT, int CT>
__device__ __forceinline__ void add_large(const v4i (&d)[RT][CT], const StagedLds<FMT, F16S, RT, CT>& l, uint32_t block, uint32_t wave,
                                          uint32_t lane, float (&acc)[RT][CT][4]) {
#pragma clang fp contract(off)
    constexpr bool kOffset = FMT == VKML_Q4_1 || FMT == VKML_Q4_K;
    const uint32_t g = lane / 16, li = lane % 16;
    float sb[CT], nsb[CT], ob[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        sb[c] = l.sb[block][16 * CT * wave + 16 * c + li];
        nsb[c] = -kSumBias * sb[c];
        ob[c] = 0.0f;
        if constexpr (kOffset) ob[c] = l.ob[block][16 * CT * wave + 16 * c + li];
    }
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const float4 sa4 = *reinterpret_cast<const float4*>(&l.sa[block][16 * r + 4 * g]);
        float4 as4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if constexpr (kOffset) as4 = *reinterpret_cast<const float4*>(&l.asum[block][16 * r + 4 * g]);
        const float sa[4] = {sa4.x, sa4.y, sa4.z, sa4.w}, asum[4] = {as4.x, as4.y, as4.z, as4.w};
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[r][c][i] += block_term<FMT, F16S>(d[r][c][i], sa[i], asum[i], sb[c], nsb[c], ob[c]);
    }
}

template <int FMT, bool F16S, int RT, int CT>
__device__ __forceinline__ void staged_load(const MatmulDotArgs& p, uint32_t t, uint32_t c0, uint32_t row0, uint32_t col0,
                                            StagedChunk<FMT, F16S, RT, CT>& r) {
    using S = StagedChunk<FMT, F16S, RT, CT>;
    constexpr uint32_t AB = S::kABlocks, kPerRow = kChunk / AB;  // threads a row
    const uint32_t blocks = p.k / 32;
    if (S::kAThreads == kT || t < S::kAThreads) {
        // A: row t / kPerRow, blocks AB (t % kPerRow) .. of the chunk
        const uint32_t row = min(row0 + t / kPerRow, p.m - 1);
#pragma unroll
        for (uint32_t h = 0; h < AB; ++h) {
            const uint32_t b = AB * (t % kPerRow) + h, blk = min(c0 + b, blocks - 1);
            const uint4* src = reinterpret_cast<const uint4*>(p.a + static_cast<uint64_t>(row) * p.k + blk * 32);
            r.a[2 * h] = ldg(src);
            r.a[2 * h + 1] = ldg(src + 1);
            r.sa[h] = ldg(p.a_scales + static_cast<uint64_t>(row) * blocks + blk);
        }
    }
    // B: 16-byte pieces of the columns' chunk bytes, consecutive threads along a column
#pragma unroll
    for (uint32_t u = 0; u < S::kBLoads; ++u) {
        const uint32_t e = t + kT * u, cl = e / (S::kBBytes / 16), piece = e % (S::kBBytes / 16);
        const uint32_t col = min(col0 + cl, p.n - 1);
        const uint8_t* src;
        if constexpr (FMT == VKML_Q8_0) {
            const uint32_t blk = min(c0 + piece / 2, blocks - 1);
            src = p.b + static_cast<uint64_t>(col) * p.k + blk * 32 + 16 * (piece % 2);
        } else if constexpr (FMT == VKML_Q4_K) {
            src = p.b + static_cast<uint64_t>(col) * (p.k / 2) + (c0 / 8) * 128 + 16 * piece;
        } else {
            const uint32_t blk = min(c0 + piece, blocks - 1);
            src = p.b + static_cast<uint64_t>(col) * (p.k / 2) + blk * 16;
        }
        r.b[u] = ldg(reinterpret_cast<const uint4*>(src));
    }
    if (S::kSThreads == kT || t < S::kSThreads) {
#pragma unroll
        for (uint32_t u = 0; u < S::kSCols; ++u) {
            const uint32_t col = min(col0 + t / 2 + kT / 2 * u, p.n - 1), b0 = 4 * (t % 2);
            if constexpr (FMT == VKML_Q4_K) {
                r.header[u] = ldg(reinterpret_cast<const uint4*>(static_cast<const uint8_t*>(p.b_scales) +
                                                                 (static_cast<uint64_t>(col) * (p.k / 256) + c0 / 8) * 16));
            } else {
#pragma unroll
                for (uint32_t b = 0; b < 4; ++b) b_block_scale<FMT, F16S>(p, col, min(c0 + b0 + b, blocks - 1), r.s[u][b], r.o[u][b]);
            }
        }
    }
}

template <int FMT, bool F16S, int RT, int CT, bool MASK>
__device__ __forceinline__ void staged_store(const StagedChunk<FMT, F16S, RT, CT>& r, uint32_t t, uint32_t left, StagedLds<FMT, F16S, RT, CT>& l) {
    using S = StagedChunk<FMT, F16S, RT, CT>;
    constexpr bool kOffset = S::kOffset;
    constexpr uint32_t AB = S::kABlocks, kPerRow = kChunk / AB;
    if (S::kAThreads == kT || t < S::kAThreads) {
        const uint32_t row = t / kPerRow;
#pragma unroll
        for (uint32_t i = 0; i < 2 * AB; ++i)
            *reinterpret_cast<uint4*>(l.a + row * S::kAStride + (t % kPerRow) * 32 * AB + 16 * i) = r.a[i];
#pragma unroll
        for (uint32_t h = 0; h < AB; ++h) {
            const uint32_t b = AB * (t % kPerRow) + h;
            // MASK: blocks past K (the last chunk of a K of other than whole
            // chunks, whose blocks are scaled in groups) re-read its last one
            // with zero scales, offsets and code sums: their terms are zeros,
            // which change no accumulator (none is ever -0).
            l.sa[b][row] = !MASK || b < left ? r.sa[h] : 0.0f;
            if constexpr (kOffset) l.asum[b][row] = !MASK || b < left ? static_cast<float>(byte_sum(r.a[2 * h]) + byte_sum(r.a[2 * h + 1])) : 0.0f;
        }
    }
#pragma unroll
    for (uint32_t u = 0; u < S::kBLoads; ++u) {
        const uint32_t e = t + kT * u, cl = e / (S::kBBytes / 16), piece = e % (S::kBBytes / 16);
        *reinterpret_cast<uint4*>(l.b + cl * S::kBStride + 16 * piece) = r.b[u];
    }
    if (S::kSThreads == kT || t < S::kSThreads) {
#pragma unroll
        for (uint32_t u = 0; u < S::kSCols; ++u) {
            const uint32_t cl = t / 2 + kT / 2 * u, b0 = 4 * (t % 2);
#pragma unroll
            for (uint32_t b = 0; b < 4; ++b) {
                float sv = r.s[u][b], ov = r.o[u][b];
                if constexpr (FMT == VKML_Q4_K) q4k_block_scale(r.header[u], b0 + b, sv, ov);
                l.sb[b0 + b][cl] = !MASK || b0 + b < left ? sv : 0.0f;
                if constexpr (kOffset) l.ob[b0 + b][cl] = !MASK || b0 + b < left ? ov : 0.0f;
            }
        }
    }
}

// Column cl's operand for block b of the staged chunk: its 8 codes at values
// 8 g .. 8 g + 7, as int8 (q4: codes 0 .. 15, or minus 8 for q4_0).
template <int FMT, bool F16S, int RT, int CT>
__device__ __forceinline__ long staged_b(const StagedLds<FMT, F16S, RT, CT>& l, uint32_t cl, uint32_t b, uint32_t g) {
    using S = StagedChunk<FMT, F16S, RT, CT>;
    const uint8_t* col = l.b + cl * S::kBStride;
    uint32_t lo, hi;
    if constexpr (FMT == VKML_Q8_0) {
        const uint2 w = *reinterpret_cast<const uint2*>(col + b * 32 + 8 * g);
        lo = w.x;
        hi = w.y;
    } else if constexpr (FMT == VKML_Q4_K) {
        const uint2 w = *reinterpret_cast<const uint2*>(col + 32 * (b / 2) + 8 * g);
        const uint32_t sh = 4 * (b % 2);
        lo = (w.x >> sh) & 0x0F0F0F0Fu;
        hi = (w.y >> sh) & 0x0F0F0F0Fu;
    } else {
        const uint32_t q = *reinterpret_cast<const uint32_t*>(col + b * 16 + 4 * g);
        if constexpr (FMT == VKML_Q4_0) {
            lo = q4_signed(q, 0);
            hi = q4_signed(q, 4);
        } else {
            lo = q & 0x0F0F0F0Fu;
            hi = (q >> 4) & 0x0F0F0F0Fu;
        }
    }
    return static_cast<long>((static_cast<uint64_t>(hi) << 32) | lo);
}

// TAIL: what the last chunk of K does (rules.hpp).
template <int FMT, bool F16S, int RT, int CT, int TAIL>
__global__ void __launch_bounds__(kT, RT * CT == 4 ? 4 : 1) k_matmul_dot(MatmulDotArgs p) {
    using S = StagedChunk<FMT, F16S, RT, CT>;
    constexpr bool kOffset = S::kOffset;
    constexpr int G = RT * CT >= 4 ? 1 : 4 / (RT * CT);  // blocks whose scaling runs together
    // (q4_K's K is whole chunks; its tiles with the masks left out are 2 to 7%
    // slower, as the compiler then orders their staging: 512 x 4096 x 4096
    // 49.6, 52.0 us)
    constexpr bool kMask = FMT == VKML_Q4_K ? RT * CT != 8 : TAIL == kMaskedTail || (TAIL == kCutTail && G > 1);
    __shared__ StagedLds<FMT, F16S, RT, CT> l;
    const uint32_t t = thread_index(), lane = t % kWave, wave = t / kWave;
    const uint32_t g = lane / 16, li = lane % 16;
    uint32_t tile_row = blockIdx.y, tile_col = blockIdx.x;
    if (p.bands.width != 0 && !p.bands.tile(blockIdx.x, tile_row, tile_col)) return;
    const uint32_t row0 = tile_row * S::TM, col0 = tile_col * S::TN;
    const uint32_t blocks = p.k / 32;
    float acc[RT][CT][4];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[r][c][i] = 0.0f;
    // A block's matrix instructions (RT x CT of them) into d.
    const auto sums = [&](uint32_t b, v4i (&d)[RT][CT]) {
        long av[RT], bv[CT];
#pragma unroll
        for (int r = 0; r < RT; ++r) av[r] = *reinterpret_cast<const long*>(l.a + (16 * r + li) * S::kAStride + b * 32 + 8 * g);
#pragma unroll
        for (int c = 0; c < CT; ++c) bv[c] = staged_b<FMT, F16S, RT, CT>(l, 16 * CT * wave + 16 * c + li, b, g);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int c = 0; c < CT; ++c) d[r][c] = __builtin_amdgcn_mfma_i32_16x16x32_i8(av[r], bv[c], sum_start<FMT, F16S>(), 0, 0, 0);
    };
    const auto stats = [&](uint32_t b, BlockStats<RT, CT>& st) {
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const uint32_t cl = 16 * CT * wave + 16 * c + li;
            st.sb[c] = l.sb[b][cl];
            st.nsb[c] = -kSumBias * st.sb[c];
            st.ob[c] = 0.0f;
            if constexpr (kOffset) st.ob[c] = l.ob[b][cl];
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            st.sa[r] = *reinterpret_cast<const float4*>(&l.sa[b][16 * r + 4 * g]);
            st.asum[r] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if constexpr (kOffset) st.asum[r] = *reinterpret_cast<const float4*>(&l.asum[b][16 * r + 4 * g]);
        }
    };
    StagedChunk<FMT, F16S, RT, CT> next;
    staged_load<FMT, F16S, RT, CT>(p, t, 0, row0, col0, next);
    for (uint32_t c0 = 0; c0 < blocks; c0 += kChunk) {
        __syncthreads();  // the last chunk's readers are done
        staged_store<FMT, F16S, RT, CT, kMask>(next, t, blocks - c0, l);
        __syncthreads();
        if (c0 + kChunk < blocks) staged_load<FMT, F16S, RT, CT>(p, t, c0 + kChunk, row0, col0, next);  // in flight meanwhile
#pragma unroll
        for (uint32_t b = 0; b < kChunk; b += G) {
            // (in the largest tile this also keeps the next block's reads, and
            // their registers, out of this one)
            if (TAIL == kCutTail && c0 + b >= blocks) break;
            if constexpr (RT * CT == 8) {
                v4i d[RT][CT];
                sums(b, d);
                add_large<FMT, F16S, RT, CT>(d, l, b, wave, lane, acc);
            } else {
                v4i d[G][RT][CT];
                BlockStats<RT, CT> st[G];
#pragma unroll
                for (int q = 0; q < G; ++q) {
                    sums(b + q, d[q]);
                    stats(b + q, st[q]);
                }
                add_tiles<FMT, F16S, RT, CT, G>(d, st, l, b, wave, lane, acc);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const uint32_t col = col0 + 16 * CT * wave + 16 * c + li;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t row = row0 + 16 * r + 4 * g + i;
                if (row < p.m && col < p.n) store_out(p, row, col, acc[r][c][i]);
            }
        }
}

template <int FMT, bool F16S, int RT, int CT>
void launch_tile(MatmulDotArgs p) {
    p.bands = dot_bands((p.m + 16 * RT - 1) / (16 * RT), (p.n + 64 * CT - 1) / (64 * CT));
    const dim3 grid = p.bands.width != 0 ? dim3(8 * p.bands.share) : dim3(p.bands.columns, p.bands.rows);
    const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kT), 0, vkml::abi::stream(), p); };
    const DotTail tail = dot_tail(RT, CT, p.k);
    if constexpr (RT * CT == 8) {
        go(k_matmul_dot<FMT, F16S, RT, CT, kCutTail>);
    } else if constexpr (FMT == VKML_Q4_K) {  // (its K is whole chunks)
        go(k_matmul_dot<FMT, F16S, RT, CT, kWholeTail>);
    } else {
        if constexpr (RT * CT == 1) {
            if (tail == kMaskedTail) return go(k_matmul_dot<FMT, F16S, RT, CT, kMaskedTail>);
        }
        tail == kWholeTail ? go(k_matmul_dot<FMT, F16S, RT, CT, kWholeTail>) : go(k_matmul_dot<FMT, F16S, RT, CT, kCutTail>);
    }
}

template <int FMT, bool F16S>
void launch(const MatmulDotArgs& p) {
    const DotTile tile = dot_tile(FMT, F16S, p.m, p.n);
    if constexpr (dot_has_64_rows(FMT)) {
        if (tile.rt == 4) return launch_tile<FMT, F16S, 4, 2>(p);
    }
    if constexpr (FMT != VKML_Q8_0) {
        if (tile.rt == 1 && tile.ct == 2) return launch_tile<FMT, F16S, 1, 2>(p);
    }
    tile.rt == 2 ? launch_tile<FMT, F16S, 2, 2>(p) : launch_tile<FMT, F16S, 1, 1>(p);
}

int matmul_dot_common(const char* what, const vkml_gemv_dot_params* p, const void* a_values, const void* b_values, float* out,
                      const void* b_scales, const float* a_scales, const float* residual) {
    VKML_REQUIRE_INIT();
    const std::string name = what;
    VKML_CHECK_ARG(p, name + ": null params");
    VKML_CHECK_ARG(p->b_type == VKML_Q8_0 || p->b_type == VKML_Q4_0 || p->b_type == VKML_Q4_1 || p->b_type == VKML_Q4_K,
                   name + ": weights must be q8_0, q4_0, q4_1 or q4_K, got type " + std::to_string(p->b_type));
    VKML_CHECK_ARG(p->b_type == VKML_Q4_K || p->scale_type == VKML_F16 || p->scale_type == VKML_F32, name + ": scales must be f16 or f32");
    const uint32_t unit = p->b_type == VKML_Q4_K ? 256 : 32;
    VKML_CHECK_ARG(p->k > 0 && p->k % unit == 0, name + ": k = " + std::to_string(p->k) + " must be a positive multiple of " + std::to_string(unit));
    if (p->m == 0 || p->n == 0) return VKML_OK;
    VKML_CHECK_ARG(a_values && b_values && out && b_scales && a_scales, name + ": null buffer");
    const MatmulDotArgs args{static_cast<const uint8_t*>(a_values), a_scales, static_cast<const uint8_t*>(b_values), b_scales, out,
                             p->m, p->n, p->k, residual, {}};
    vkml::abi::ProfileScope prof(what);
    const bool f16 = p->scale_type == VKML_F16;
    switch (p->b_type) {
        case VKML_Q8_0: f16 ? launch<VKML_Q8_0, true>(args) : launch<VKML_Q8_0, false>(args); break;
        case VKML_Q4_0: f16 ? launch<VKML_Q4_0, true>(args) : launch<VKML_Q4_0, false>(args); break;
        case VKML_Q4_1: f16 ? launch<VKML_Q4_1, true>(args) : launch<VKML_Q4_1, false>(args); break;
        default: launch<VKML_Q4_K, true>(args); break;
    }
    return vkml::abi::check_launch(what);
}

}  // namespace

extern "C" {

int vkml_matmul_dot(const vkml_gemv_dot_params* p, const void* a_values, const void* b_values, float* out, const void* b_scales,
                    const float* a_scales) {
    return matmul_dot_common("matmul_dot", p, a_values, b_values, out, b_scales, a_scales, nullptr);
}

int vkml_matmul_dot_add(const vkml_gemv_dot_params* p, const void* a_values, const void* b_values, float* out, const void* b_scales,
                        const float* a_scales, const float* residual) {
    VKML_REQUIRE_INIT();
    VKML_CHECK_ARG(residual || (p && (p->m == 0 || p->n == 0)), "matmul_dot_add: null residual");
    return matmul_dot_common("matmul_dot_add", p, a_values, b_values, out, b_scales, a_scales, residual);
}

}  // extern "C"
