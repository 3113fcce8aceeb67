// k_matmul_f32.hip -- the f32 matrix product of many rows (prefill): the
// reference's shaders/matmul.comp (src/ops/matmul.cpp:44-120), attention's
// scores and probs v and the float path's projections.
//
// Order (matmul.comp:131-140). Every output sums a[m][k] * b(k, n) in k
// order, a product and an add at a time, each rounded to f32. The adds are a
// chain per output and stay on the VALU; the products are outer products of
// a column of a and a row of b, and v_mfma_f32_16x16x1_4b_f32 with a zero
// accumulator forms 1024 of them at once, each rounded once (fma(a, b, 0)):
// the bits of the VALU's product, subnormals included. (A product of -0
// comes out +0; no sum that starts at +0 can tell.)
//
// What bounds it. The add of every product: a SIMD with waves enough issues a
// wave64 add about every 1.04 ns, and the matrix unit, which does not run
// beside the VALU, takes 0.85 ns for a lane's product: 1.9 ns for the two at
// best, 34.6 T multiply-accumulates a second over the GPU (a loop of nothing
// else reaches 31.5), of which the large products reach 30. The kernel before
// it, 4 x 4 outputs a thread with a multiply and an add each, read 512 lane
// values from LDS for a wave's 1024 products, where a wave here reads 192 for
// 2048, and reached 20 to 26. Measured before and after (us; f16 b): probs v of
// 2048 queries by 4096 keys, 32 heads of 128, 1287 -> 915, its scores 1152 ->
// 912; 512 queries from position 0 60 -> 26 and 46 -> 29; 200 x 8192 x 2048
// 209 -> 154, 200 x 2048 x 8192 863 -> 218. A quantized b's codes are widened
// when they are staged (q4_K 512 x 4096 x 4096 719 -> 384).
//
// Registers. Four waves a SIMD; the element-load forms of an f32 b and three
// 32-row tiles of quantized ones spill up to nine registers for it. With three
// waves and none spilled they are equal or up to 3% slower (2000 x 8193 x 1025,
// f32 b by elements, 694, 704 us).
//
// Mapping. A wave computes 16 NC rows by 16 R columns; one instruction's
// four 16 x 16 blocks are R column blocks by 4 / R consecutive k's, so that
// short products get smaller tiles with the same work an instruction, and b
// is its first operand, so that a lane's results are four columns of a row
// (one 16-byte store). K runs in chunks staged in LDS as f32, the next
// chunk's global loads in flight in registers meanwhile; a row of the staged
// a (and of a transposed b) holds its k's grouped by the block that
// multiplies them, so a lane reads four steps' operands with one 16-byte
// load. The adds trail one instruction behind, so that the matrix unit's
// latency is covered.
#include <algorithm>

#include "device.hpp"
#include "internal.hpp"
#include "rules.hpp"

// Products and sums are rounded apart.
#pragma clang fp contract(off)

using namespace vkml::dev;
using vkml::abi::ProfileScope;
using namespace vkml::rules;

namespace {

constexpr uint32_t kT = 256;   // four waves
typedef float v16f __attribute__((ext_vector_type(16)));

struct MatmulArgs {
    vkml_matmul_params p;
    const float* a;
    const void* b;
    const void* bs;
    float* c;
    uint32_t vec_c;  // c's rows are whole, aligned vec4s
};

// Four elements of b as stored, along its rows (so of one block of a
// quantized b): floats; or the codes' word and their scale and offset, f16 or
// f32 bits, or q4_K header. They are widened when they are staged, so that a
// chunk's loads wait for nothing.
template <uint32_t BTYPE>
struct BRaw {
    uint32_t codes, scale, offset;
};
template <>
struct BRaw<VKML_Q4_K> {
    uint32_t codes;
    uint4 header;
};
template <>
struct BRaw<VKML_F32> {
    float4 v;
};
template <>
struct BRaw<VKML_F16> {
    uint2 v;
};
template <>
struct BRaw<VKML_BF16> {
    uint2 v;
};

// Elements col .. col + 3 (col a multiple of 4) of row `row` of a quantized b
// [rows, cols].
template <uint32_t BTYPE>
__device__ __forceinline__ BRaw<BTYPE> load_codes(const MatmulArgs& g, uint64_t row, uint32_t col) {
    const uint64_t cols = g.p.k, e = row * cols + col;
    BRaw<BTYPE> r{};
    if constexpr (BTYPE == VKML_Q4_K) {
        // sub-block j of the super-block: the low or the high nibbles of bytes 32 (j / 2) ..
        const uint32_t j = col % 256 / 32;
        __builtin_memcpy(&r.codes, static_cast<const uint8_t*>(g.b) + row * (cols / 2) + col / 256 * 128 + 32 * (j / 2) + col % 32, 4);
        r.header = static_cast<const uint4*>(g.bs)[row * (cols / 256) + col / 256];
    } else {
        if constexpr (BTYPE == VKML_Q8_0) __builtin_memcpy(&r.codes, static_cast<const uint8_t*>(g.b) + e, 4);
        else r.codes = static_cast<const uint32_t*>(g.b)[e / 8];
        constexpr uint32_t per = BTYPE == VKML_Q4_1 ? 2 : 1;
        const uint64_t at = e / 32 * per;
        if (g.p.scale_type == VKML_F16) {
            r.scale = static_cast<const uint16_t*>(g.bs)[at];
            if constexpr (per == 2) r.offset = static_cast<const uint16_t*>(g.bs)[at + 1];
        } else {
            r.scale = static_cast<const uint32_t*>(g.bs)[at];
            if constexpr (per == 2) r.offset = static_cast<const uint32_t*>(g.bs)[at + 1];
        }
    }
    return r;
}

// The four elements' values (weight_value's), col their place in the row.
template <uint32_t BTYPE>
__device__ __forceinline__ float4 widen(const BRaw<BTYPE>& w, uint32_t col, uint32_t scale_type) {
    if constexpr (BTYPE == VKML_F32) {
        return w.v;
    } else if constexpr (BTYPE == VKML_F16 || BTYPE == VKML_BF16) {
        return make_float4(half_to_float(w.v.x & 0xFFFFu, BTYPE), half_to_float(w.v.x >> 16, BTYPE), half_to_float(w.v.y & 0xFFFFu, BTYPE),
                           half_to_float(w.v.y >> 16, BTYPE));
    } else {
        float s, o = 0.0f, v[4];
        if constexpr (BTYPE == VKML_Q4_K) {
            q4k_block_scale(w.header, col % 256 / 32, s, o);
        } else {
            s = scale_type == VKML_F16 ? f16_bits_to_float(static_cast<uint16_t>(w.scale)) : __uint_as_float(w.scale);
            if constexpr (BTYPE == VKML_Q4_1) o = scale_type == VKML_F16 ? f16_bits_to_float(static_cast<uint16_t>(w.offset)) : __uint_as_float(w.offset);
        }
        const uint32_t half = BTYPE == VKML_Q4_K ? col % 64 / 32 : col % 8 / 4;  // low or high nibbles
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            if constexpr (BTYPE == VKML_Q8_0) {
                v[i] = static_cast<float>(static_cast<int8_t>(w.codes >> (8 * i))) * s;
            } else {
                const uint32_t q = (w.codes >> (8 * i + 4 * half)) & 15u;
                if constexpr (BTYPE == VKML_Q4_0) v[i] = static_cast<float>(static_cast<int>(q) - 8) * s;
                else v[i] = static_cast<float>(q) * s + o;
            }
        }
        return make_float4(v[0], v[1], v[2], v[3]);
    }
}

// v with the elements from i on that are not below end set to zero.
__device__ __forceinline__ float4 keep_below(float4 v, uint32_t i, uint32_t end) {
    return make_float4(i < end ? v.x : 0.0f, i + 1 < end ? v.y : 0.0f, i + 2 < end ? v.z : 0.0f, i + 3 < end ? v.w : 0.0f);
}

// Under a causal mask: how many column tiles hold keys that row tile ty sees.
__host__ __device__ __forceinline__ uint32_t visible_tiles(const vkml_matmul_params& p, uint32_t ty, uint32_t tm, uint32_t tn) {
    const uint64_t last_key = static_cast<uint64_t>(ty) * tm + tm - 1 + p.causal_offset;
    return static_cast<uint32_t>(last_key < p.n - 1 ? last_key : p.n - 1) / tn + 1;
}

template <bool BT, uint32_t BTYPE, int R, int NC, int LOADS, bool CUT>
__global__ void __launch_bounds__(kT, 4) k_matmul(MatmulArgs g) {
    constexpr uint32_t KK = 4 / R;                 // k's an instruction
    constexpr uint32_t WR = R == 1 ? 1 : 2;        // waves along the rows
    constexpr uint32_t TM = 16 * NC * WR, TN = 16 * R * (4 / WR);  // the workgroup's tile
    constexpr uint32_t kKB = R == 1 ? 64 : 32;     // k's a chunk
    constexpr uint32_t kStr = kKB + 4;             // floats a staged row: 16-byte reads of 16 rows hit every bank once
    constexpr uint32_t PK = kKB / KK;              // k's of a chunk a block multiplies
    constexpr uint32_t kBStr = TN + 16;            // b [k, n] staged: KK rows hit different banks
    constexpr uint32_t kAThreads = TM * kKB / 4 < kT ? TM * kKB / 4 : kT;
    constexpr uint32_t NA = TM * kKB / 4 / kAThreads, NB = TN * kKB / 4 / kT;  // vec4 loads a thread
    __shared__ __align__(16) float ta[TM * kStr];
    __shared__ __align__(16) float tb[BT ? TN * kStr : kKB * kBStr];
    const vkml_matmul_params& p = g.p;
    const uint32_t t = threadIdx.x, lane = t % kWave, wave = t / kWave, li = lane % 16, blk = lane / 16;
    const uint32_t wave_m = 16 * NC * (wave % WR), wave_n = 16 * R * (wave / WR);  // the wave's tile in it
    // blockIdx: column tile, batch, row tile. Under a causal mask the later
    // rows of probs v do the most: they start first, of every batch, so each
    // compute unit gets its share of long and short ones. The scores a mask
    // leaves are a staircase of tiles: row tiles from both ends are paired,
    // so that every pair launches about as many tiles and few workgroups
    // have nothing to do (a launch over every column tile, whose empty ones
    // fall on some XCDs more than on others, gained nothing from the mask:
    // 1185 us at 2048 queries by 4096 keys, 1230 without it).
    uint32_t ty = !BT && p.causal ? gridDim.z - 1 - blockIdx.z : blockIdx.z, tx = blockIdx.x;
    if (BT && p.causal) {
        const uint32_t rows = (p.m + TM - 1) / TM, other = rows - 1 - ty, n = visible_tiles(p, other, TM, TN);
        if (tx < n) {
            ty = other;
        } else {
            tx -= n;
            if (ty == other || tx >= visible_tiles(p, ty, TM, TN)) return;
        }
    }
    const uint32_t row0 = ty * TM, col0 = tx * TN, z = blockIdx.y;
    // The tile's last row sees keys up to row0 + TM - 1 + offset: scores
    // past it are never read, and a's entries past it are 0.
    const uint64_t last_key = static_cast<uint64_t>(row0) + TM - 1 + p.causal_offset;
    const uint32_t k_end = (!BT && p.causal) ? static_cast<uint32_t>(min<uint64_t>(p.k, last_key + 1)) : p.k;
    // A wave with nothing to compute still stages, for the others.
    const bool idle = col0 + wave_n >= p.n || row0 + wave_m >= p.m || (BT && p.causal && col0 + wave_n > last_key);
    // The operands: a's rows from row0, b's batch.
    const float* a0 = g.a + (static_cast<uint64_t>(z) * p.m + row0) * p.k;
    const uint64_t b0 = static_cast<uint64_t>(z / p.b_group) * p.b_stride + (BT ? static_cast<uint64_t>(col0) * p.k : 0);
    using Off = std::conditional_t<LOADS == kVecAB, uint32_t, uint64_t>;
    constexpr bool kChunkBase = !BT && LOADS == kVecAB;  // offsets of a b [k, n] from the chunk's first row

    // Every load of a chunk is issued without a branch (indices past the
    // operands re-read their last elements: rows and columns past the end
    // are not stored, and store() clears the k's past k_end), so that nothing
    // waits for them before store().
    float4 ra[NA];
    BRaw<BTYPE> rb[NB];
    const auto load = [&](uint32_t k0) {
        if (kAThreads == kT || t < kAThreads) {
#pragma unroll
            for (uint32_t u = 0; u < NA; ++u) {
                const uint32_t e = t + kT * u, row = min(e / (kKB / 4), p.m - 1 - row0), k = k0 + 4 * (e % (kKB / 4));
                const Off at = static_cast<Off>(row) * p.k;
                if constexpr (LOADS == kVecAB) {
                    ra[u] = *reinterpret_cast<const float4*>(a0 + (at + min(k, p.k - 4)));
                } else {
                    const float* src = a0 + at;
                    ra[u] = make_float4(src[min(k, p.k - 1)], src[min(k + 1, p.k - 1)], src[min(k + 2, p.k - 1)], src[min(k + 3, p.k - 1)]);
                }
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < NB; ++u) {
            const uint32_t e = t + kT * u;
            // four elements along the rows of b: `from` of a row of `len`, the
            // tile's row `line` (of a b [k, n] the chunk's, or b's)
            const uint32_t line0 = BT || kChunkBase ? 0 : k0;
            const uint32_t line = BT ? min(e / (kKB / 4), p.n - 1 - col0) : min(line0 + e / (TN / 4), p.k - 1 - (k0 - line0));
            const uint32_t from = BT ? k0 + 4 * (e % (kKB / 4)) : col0 + 4 * (e % (TN / 4)), len = BT ? p.k : p.n;
            if constexpr (BTYPE >= VKML_Q8_0) {
                rb[u] = load_codes<BTYPE>(g, col0 + line, min(from, p.k - 4));
            } else {
                using E = std::conditional_t<BTYPE == VKML_F32, float, uint16_t>;
                const E* base = static_cast<const E*>(g.b) + b0 + (kChunkBase ? static_cast<uint64_t>(k0) * p.n : 0);
                const Off at = static_cast<Off>(line) * len;
                if constexpr (LOADS != kScalar) {
                    rb[u].v = *reinterpret_cast<const decltype(rb[u].v)*>(base + (at + min(from, len - 4)));
                } else {
                    const E* src = base + at;
                    const E e0 = src[min(from, len - 1)], e1 = src[min(from + 1, len - 1)], e2 = src[min(from + 2, len - 1)], e3 = src[min(from + 3, len - 1)];
                    if constexpr (BTYPE == VKML_F32) rb[u].v = make_float4(e0, e1, e2, e3);
                    else rb[u].v = make_uint2(e0 | (static_cast<uint32_t>(e1) << 16), e2 | (static_cast<uint32_t>(e3) << 16));
                }
            }
        }
    };
    // Four k's of a staged row: k at [k % KK][k / KK].
    const auto put = [](float* row, uint32_t kq, float4 v) {
        if constexpr (KK == 1) {
            *reinterpret_cast<float4*>(row + 4 * kq) = v;
        } else if constexpr (KK == 2) {
            *reinterpret_cast<float2*>(row + 2 * kq) = make_float2(v.x, v.z);
            *reinterpret_cast<float2*>(row + PK + 2 * kq) = make_float2(v.y, v.w);
        } else {
            row[kq] = v.x;
            row[PK + kq] = v.y;
            row[2 * PK + kq] = v.z;
            row[3 * PK + kq] = v.w;
        }
    };
    const auto store = [&](uint32_t k0) {
        const bool tail = k0 + kKB > k_end;
        if (kAThreads == kT || t < kAThreads) {
#pragma unroll
            for (uint32_t u = 0; u < NA; ++u) {
                const uint32_t e = t + kT * u, kq = e % (kKB / 4);
                put(ta + (e / (kKB / 4)) * kStr, kq, tail ? keep_below(ra[u], k0 + 4 * kq, k_end) : ra[u]);
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < NB; ++u) {
            const uint32_t e = t + kT * u;
            const float4 v = widen<BTYPE>(rb[u], BT ? k0 + 4 * (e % (kKB / 4)) : 0, p.scale_type);
            if constexpr (BT) {
                const uint32_t kq = e % (kKB / 4);
                put(tb + (e / (kKB / 4)) * kStr, kq, tail ? keep_below(v, k0 + 4 * kq, k_end) : v);
            } else {
                const uint32_t k = e / (TN / 4);
                *reinterpret_cast<float4*>(tb + k * kBStr + 4 * (e % (TN / 4))) = tail && k0 + k >= k_end ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : v;
            }
        }
    };

    // Block blk of an instruction: b's column block blk % R (the rows of the
    // matrix unit's result) by a's rows, at its k number blk / R. A lane gets
    // four columns in a row of c.
    const uint32_t kk = blk / R;
    const float* a_at = ta + (wave_m + li) * kStr + kk * PK;
    const float* b_at = BT ? tb + (wave_n + 16 * (blk % R) + li) * kStr + kk * PK : tb + kk * kBStr + wave_n + 16 * (blk % R) + li;
    float acc[NC][R][4];
    const auto add = [&](int c, const v16f& d) {
#pragma unroll
        for (uint32_t k = 0; k < KK; ++k)
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[c][r][i] += d[4 * (r + R * k) + i];
    };
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[c][r][i] = 0.0f;
    v16f last{};  // the products not added yet, of row block NC - 1
    load(0);
    for (uint32_t k0 = 0; k0 < k_end; k0 += kKB) {
        __syncthreads();  // the last chunk's readers are done
        store(k0);
        __syncthreads();
        if (k0 + kKB < k_end) load(k0 + kKB);
        if (idle) continue;
        // CUT: the last chunk's k's past the sums are left out, two steps at a
        // time.
        const uint32_t end = !CUT ? PK / 4 : min(PK / 4, 2 * ((k_end - k0 + 8 * KK - 1) / (8 * KK)));
#pragma unroll 2
        for (uint32_t q = 0; q < end; ++q) {
            float av[NC][4], bv[4];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const float4 a4 = *reinterpret_cast<const float4*>(a_at + 16 * c * kStr + 4 * q);
                av[c][0] = a4.x;
                av[c][1] = a4.y;
                av[c][2] = a4.z;
                av[c][3] = a4.w;
            }
            if constexpr (BT) {
                const float4 b4 = *reinterpret_cast<const float4*>(b_at + 4 * q);
                bv[0] = b4.x;
                bv[1] = b4.y;
                bv[2] = b4.z;
                bv[3] = b4.w;
            } else {
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) bv[j] = b_at[KK * (4 * q + j) * kBStr];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const v16f d = __builtin_amdgcn_mfma_f32_16x16x1f32(bv[j], av[c][j], v16f{}, 0, 0, 0);
                    add((c + NC - 1) % NC, last);
                    last = d;
                }
        }
    }
    if (idle) return;
    add(NC - 1, last);
    float* out = g.c + (static_cast<uint64_t>(z) * p.m + row0 + wave_m) * p.n + col0 + wave_n;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const uint32_t row = 16 * c + li;
        if (row0 + wave_m + row >= p.m) continue;
        float* o = out + static_cast<uint64_t>(row) * p.n;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint32_t at = 16 * r + 4 * blk, col = col0 + wave_n + at;
            if (g.vec_c) {
                if (col < p.n) *reinterpret_cast<float4*>(o + at) = make_float4(acc[c][r][0], acc[c][r][1], acc[c][r][2], acc[c][r][3]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (col + i < p.n) o[at + i] = acc[c][r][i];
            }
        }
    }
}

template <bool BT, uint32_t BTYPE, int LOADS, int R, int NC, bool CUT = R == 4>
void launch_tile(const MatmulArgs& g) {
    constexpr uint32_t WR = R == 1 ? 1 : 2, TM = 16 * NC * WR, TN = 16 * R * (4 / WR);
    dim3 grid((g.p.n + TN - 1) / TN, g.p.batches, (g.p.m + TM - 1) / TM);
    if (BT && g.p.causal) {
        // Row tile ty sees min(keys, a line in ty) / TN tiles, so a pair sees
        // at most one more than twice the middle tile's.
        const uint32_t rows = grid.z;
        grid.x = rows == 1 ? visible_tiles(g.p, 0, TM, TN) : 2 * visible_tiles(g.p, rows / 2, TM, TN) + 1;
        grid.z = (rows + 1) / 2;
    }
    hipLaunchKernelGGL((k_matmul<BT, BTYPE, R, NC, LOADS, CUT>), grid, dim3(kT), 0, vkml::abi::stream(), g);
}

template <bool BT, uint32_t BTYPE, int LOADS>
void launch(const MatmulArgs& g) {
    const WaveTile tile = wave_tile(g.p);
    if constexpr (BTYPE != VKML_Q4_K) {
        if (tile.r == 4) return launch_tile<BT, BTYPE, LOADS, 4, 2>(g);
    }
    if constexpr (BT && BTYPE <= VKML_BF16) {
        if (tile.r == 2 && cut_last_chunk(g.p)) return tile.nc == 2 ? launch_tile<BT, BTYPE, LOADS, 2, 2, true>(g) : launch_tile<BT, BTYPE, LOADS, 2, 1, true>(g);
    }
    if (tile.r == 2) tile.nc == 2 ? launch_tile<BT, BTYPE, LOADS, 2, 2>(g) : launch_tile<BT, BTYPE, LOADS, 2, 1>(g);
    else launch_tile<BT, BTYPE, LOADS, 1, 1>(g);
}

template <uint32_t BTYPE>
void launch_float(const MatmulArgs& g) {
    const Loads loads = vkml::rules::float_loads(g.p, reinterpret_cast<uintptr_t>(g.a), reinterpret_cast<uintptr_t>(g.b));
    if (g.p.b_transposed) loads == kVecAB ? launch<true, BTYPE, kVecAB>(g) : launch<true, BTYPE, kScalar>(g);
    else if (loads == kVecAB) launch<false, BTYPE, kVecAB>(g);
    else loads == kVecB ? launch<false, BTYPE, kVecB>(g) : launch<false, BTYPE, kScalar>(g);
}

template <uint32_t BTYPE>
void launch_quant(const MatmulArgs& g) {
    quant_loads(g.p, reinterpret_cast<uintptr_t>(g.a)) == kVecAB ? launch<true, BTYPE, kVecAB>(g) : launch<true, BTYPE, kScalar>(g);
}

}  // namespace

extern "C" int vkml_matmul(const vkml_matmul_params* p, const float* a, const void* b, float* c, const void* b_scales) {
    VKML_REQUIRE_INIT();
    VKML_CHECK_ARG(p, "matmul: null params");
    VKML_CHECK_ARG(p->b_type <= VKML_Q4_K, "matmul: unknown b type " + std::to_string(p->b_type));
    VKML_CHECK_ARG(p->b_group >= 1 && p->batches >= 1, "matmul: bad batching");
    const bool quant = p->b_type >= VKML_Q8_0;
    VKML_CHECK_ARG(!p->causal || !quant, "matmul: the causal skip is for attention's products, not weights");
    if (quant) {
        VKML_CHECK_ARG(p->b_transposed && p->batches == 1, "matmul: quantized b must be one transposed [n, k] matrix");
        const uint32_t unit = p->b_type == VKML_Q4_K ? 256 : 32;
        VKML_CHECK_ARG(p->k % unit == 0, "matmul: k = " + std::to_string(p->k) + " is not whole blocks of " + std::to_string(unit));
        VKML_CHECK_ARG(p->scale_type == VKML_F16 || (p->scale_type == VKML_F32 && p->b_type != VKML_Q4_K),
                       "matmul: bad scale type");
        VKML_CHECK_ARG(b_scales, "matmul: quantized b needs scales");
    }
    if (p->m == 0 || p->n == 0) return VKML_OK;
    VKML_CHECK_ARG(a && b && c, "matmul: null buffer");
    VKML_CHECK_ARG((p->m + 63) / 64 <= 65535 && p->batches <= 65535, "matmul: too many rows or batches");
    ProfileScope prof("matmul");
    const MatmulArgs g{*p, a, b, b_scales, c, p->n % 4 == 0 && reinterpret_cast<uintptr_t>(c) % 16 == 0};
    if (p->k == 0) {
        // no products: every output is the empty sum
        return vkml_fill_u32(c, 0, static_cast<uint64_t>(p->m) * p->n * p->batches);
    }
    switch (p->b_type) {
        case VKML_F32: launch_float<VKML_F32>(g); break;
        case VKML_F16: launch_float<VKML_F16>(g); break;
        case VKML_BF16: launch_float<VKML_BF16>(g); break;
        case VKML_Q8_0: launch_quant<VKML_Q8_0>(g); break;
        case VKML_Q4_0: launch_quant<VKML_Q4_0>(g); break;
        case VKML_Q4_1: launch_quant<VKML_Q4_1>(g); break;
        default: launch_quant<VKML_Q4_K>(g); break;
    }
    return vkml::abi::check_launch("matmul");
}
