// k_prompt_fast.hip -- a prompt's causal attention on the matrix cores: the
// tolerance form of the reference's chunked q.k^T, softmax and probs.v
// (src/ops/attention.cpp:127-138,205-226), as an option beside the exact
// path (matmul scores, softmax, matmul probs.v in the reference's order).
//
// Not the reference's order of f32 operations: every product is exact (f16
// x f16 in the matrix unit, q and the probabilities split into two f16
// terms) and every sum accumulates in f32, in the matrix unit's order, with
// the softmax taken online over blocks of keys. The results are those of
// f32 attention to within f32 rounding.
//
// A workgroup takes 16 queries of one KV head's four query heads, a wave a
// head, and walks the keys its queries see in blocks of KB = 32 or 64:
//   - scores S^T [KB keys x 16 queries] = K . Q^T by
//     v_mfma_f32_16x16x32_f16, K copied into LDS a block ahead by
//     global_load_lds (each row's 16-byte pieces swizzled so that the 16
//     rows of an operand read hit different banks), q (scaled into log2
//     units) as hi + lo f16 terms;
//   - per query (a lane column) the block's max and the running (max, sum),
//     the accumulated output rescaled by 2^(m_old - m_new);
//   - O^T [hd x 16 queries] += V^T . P^T, V loaded a block ahead into
//     registers and written into LDS transposed, [dim][key], two keys a
//     word, so that a lane's operand is two 8-byte reads; P^T straight from
//     the score tile's registers (the accumulator layout of S^T is the B
//     operand's of P^T, keys permuted alike in V^T's A operand). In O^T a
//     query is a lane column, as in S^T, so its rescale needs no exchange
//     between lanes.
// The output is written [query, head, hd]: the o projection's input rows.
//
// What bounds it. A tile's blocks follow one another, and few workgroups run
// beside it: a wave's matrix instructions (64 a 64-key block at head_dim 128,
// about 0.4 us), its softmax, and the LDS and barrier waits between them take
// 2 us a block. 1000 queries after 37 keys, 32 heads on 8 KV heads of 128:
// 63.0 us with an f16 a V^T store and 32-key blocks, 43.7 with two keys a
// store and 64-key blocks, 41.0 with masks only where a tile's queries need
// them, the output rescaled only when a maximum has moved, and the sums of a
// query's four lanes added once, 37.7 with the matrix instructions of several
// tiles in turn.
#include <algorithm>
#include <string>

#include "attend_fast.hpp"
#include "device.hpp"
#include "internal.hpp"
#include "rules.hpp"

using namespace vkml::dev;
using vkml::attend::kThreads;
using vkml::attend_fast::f32x4;
using vkml::attend_fast::half8;
using vkml::attend_fast::kLog2e;

namespace {

constexpr uint32_t kQueries = 16;  // queries a workgroup
constexpr uint32_t kHeads = 4;     // query heads a workgroup (a wave each)

struct PromptArgs {
    const float* q;  // [heads, t, hd] f32
    const void* k_cache;
    const void* v_cache;  // [kv_heads, capacity, hd] f16
    float* out;           // [t, heads, hd] f32
    uint32_t heads, kv_heads, group, capacity, t, first;
    float scale, softcap;
};

// A block's tiles in LDS. K row-major, each row's 16-byte pieces swizzled
// (piece p of key row r at p ^ (r % pieces)) so that the 16 rows a score
// operand read takes hit different banks. V transposed, [dim][key] with
// rows padded to KB + 4 keys, so that a lane's four keys of one dim are one
// 8-byte read and the 16 dims of a read hit different banks.
template <int HD, int KB>
struct PromptTiles {
    static constexpr uint32_t kPieces = HD * 2 / 16;  // 16-byte pieces a key row
    static constexpr uint32_t kVtStride = KB + 4;      // f16 a V^T row
    alignas(16) uint8_t k[KB * HD * 2];
    alignas(16) _Float16 vt[HD * kVtStride];
};

// V of the next block in registers, 8 dims of two consecutive keys an item.
// An item's wave covers 16 key pairs by 4 pieces of 8 dims: in V^T, whose
// rows are 18 or 34 words, those 64 lanes' words (a key pair of one dim) lie
// in 64 different banks. (One key a lane and item, an f16 a store, took
// twice as many stores and four lanes a bank.)
template <int HD, int KB>
struct VRegs {
    static constexpr uint32_t kGroups = (KB / 32) * (HD / 32);  // (16 key pairs, 4 pieces) groups
    static constexpr uint32_t kWaves = kThreads / kWave;
    static constexpr uint32_t kItems = (kGroups + kWaves - 1) / kWaves;
    uint4 v[kItems][2];
    __device__ static uint32_t group(uint32_t i) { return i * kWaves + thread_index() / kWave; }
    __device__ static uint32_t pair(uint32_t i) { return group(i) / (HD / 32) * 16 + thread_index() % 16; }
    __device__ static uint32_t piece(uint32_t i) { return group(i) % (HD / 32) * 4 + thread_index() % kWave / 16; }
};

// Key block kb's K rows into LDS (global_load_lds, swizzled) and its V rows
// into registers. Keys past `keys` re-read the last.
template <int HD, int KB>
__device__ __forceinline__ void load_block(const PromptArgs& a, uint32_t kvh, uint32_t kb, uint32_t keys, PromptTiles<HD, KB>& tl,
                                           VRegs<HD, KB>& vr) {
    using T = PromptTiles<HD, KB>;
    using V = VRegs<HD, KB>;
    constexpr uint32_t RB = HD * 2;
    const uint32_t t = thread_index(), wave_first = t - t % kWave;
    const uint64_t row0 = static_cast<uint64_t>(kvh) * a.capacity;
    const auto* kc = static_cast<const uint8_t*>(a.k_cache);
    const auto* vc = static_cast<const uint8_t*>(a.v_cache);
    const auto row_of = [&](uint32_t key) -> uint64_t { return row0 + min(kb * KB + key, keys - 1); };
#pragma unroll
    for (uint32_t i = 0; i < KB * RB / 16 / kThreads; ++i) {
        const uint32_t u = i * kThreads + t, rr = u / T::kPieces, piece = u % T::kPieces;
        vkml::attend::load_to_lds16(kc + row_of(rr) * RB + 16 * (piece ^ (rr % T::kPieces)), tl.k + 16 * (i * kThreads + wave_first));
    }
#pragma unroll
    for (uint32_t i = 0; i < V::kItems; ++i) {
        if (V::group(i) >= V::kGroups) break;
#pragma unroll
        for (uint32_t e = 0; e < 2; ++e)
            vr.v[i][e] = ldg(reinterpret_cast<const uint4*>(vc + row_of(2 * V::pair(i) + e) * RB + 16 * V::piece(i)));
    }
}

// The block's V from registers into its V^T tile.
template <int HD, int KB>
__device__ __forceinline__ void store_vt(const VRegs<HD, KB>& vr, PromptTiles<HD, KB>& tl) {
    using T = PromptTiles<HD, KB>;
    using V = VRegs<HD, KB>;
#pragma unroll
    for (uint32_t i = 0; i < V::kItems; ++i) {
        if (V::group(i) >= V::kGroups) break;
        _Float16* to = tl.vt + 8 * V::piece(i) * T::kVtStride + 2 * V::pair(i);
        const uint4 x = vr.v[i][0], y = vr.v[i][1];
        const uint32_t xs[4] = {x.x, x.y, x.z, x.w}, ys[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            *reinterpret_cast<uint32_t*>(to + 2 * e * T::kVtStride) = (xs[e] & 0xFFFFu) | (ys[e] << 16);
            *reinterpret_cast<uint32_t*>(to + (2 * e + 1) * T::kVtStride) = (xs[e] >> 16) | (ys[e] & 0xFFFF0000u);
        }
    }
}

template <int HD, int KB>
__global__ void __launch_bounds__(kThreads) k_attend_prompt_fast(PromptArgs a) {
    using T = PromptTiles<HD, KB>;
    constexpr int TT = KB / 16;  // score tiles a block
    __shared__ T s_t[2];
    constexpr int kSteps = HD / 32;
    const uint32_t t = thread_index(), w = t / kWave, l = t % kWave, j = l % 16, g = l / 16;
    // Workgroup L: (KV head, head quad) set L % sets, query tile from the
    // last down. Workgroups are dealt to the 8 XCDs round-robin, so with 8
    // (or a multiple of 8) sets each XCD serves the same KV heads and their
    // K and V stay in its L2 (a KV head's 4096 keys are 2 MiB); the tiles
    // whose queries see the most keys go first.
    const uint32_t quads = a.group / kHeads, sets = a.kv_heads * quads, tiles = (a.t + kQueries - 1) / kQueries;
    const uint32_t set = blockIdx.x % sets, tile = tiles - 1 - blockIdx.x / sets;
    const uint32_t kvh = set / quads, h = kvh * a.group + (set % quads) * kHeads + w;
    const uint32_t q0 = tile * kQueries;
    const uint32_t qi = q0 + j;                                      // the lane's query
    const bool qlive = qi < a.t;
    const uint32_t qpos = a.first + min(qi, a.t - 1);                // its position: keys 0 .. qpos
    const uint32_t keys = a.first + min(q0 + kQueries, a.t);         // keys the workgroup's queries see
    const uint32_t blocks = (keys + KB - 1) / KB;
    const bool cap = a.softcap > 0.0f;

    VRegs<HD, KB> vr;
    load_block<HD, KB>(a, kvh, 0, keys, s_t[0], vr);
    // q of the lane's query, scaled (in log2 units without a soft cap), as hi + lo f16
    half8 qh[kSteps], ql[kSteps];
    {
        const float qs = cap ? a.scale : a.scale * kLog2e;
        const float* qp = a.q + (static_cast<uint64_t>(h) * a.t + min(qi, a.t - 1)) * HD + 8 * g;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const float4 x0 = ldg(reinterpret_cast<const float4*>(qp + 32 * s));
            const float4 x1 = ldg(reinterpret_cast<const float4*>(qp + 32 * s + 4));
            const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                // The f32 product through an empty asm: both terms come from
                // this one value. Otherwise the compiler folds f16(x qs) into
                // one rounding (v_fma_mixlo_f16) for the residual while the
                // packed operand rounds the f32 product, and where the two
                // differ by an f16 ulp the residual belongs to another high
                // term.
                float v = x[e] * qs;
                asm volatile("" : "+v"(v));
                qh[s][e] = static_cast<_Float16>(v);
                ql[s][e] = static_cast<_Float16>(v - static_cast<float>(qh[s][e]));
            }
        }
    }
    f32x4 o[HD / 16];
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) o[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // The lane's query: running max (log2 units) and the sum over the lane's
    // keys (the query's four lanes' are added at the end). The max starts at
    // the lowest finite value, so that scores of -inf (masked ones among
    // them) give 2^(-inf) = 0 whatever came before.
    float m = -__FLT_MAX__, lsum = 0.0f;

    // One block: wait for its loads, put its V into the V^T tile, issue the
    // next block's loads (K into the other tile's LDS, V into registers),
    // then the scores, the online softmax and O^T. Blocks alternate between
    // the two tiles (a pair a trip, so each is named statically).
    const auto block = [&](uint32_t kb, T& cur, T& nxt) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's K copies and V loads of block kb have landed
        store_vt<HD, KB>(vr, cur);
        __syncthreads();  // every wave's; and block kb - 1's tiles are no longer read
        if (kb + 1 < blocks) load_block<HD, KB>(a, kvh, kb + 1, keys, nxt, vr);
        // scores: lane (j, g) holds keys KB kb + 16 tt + 4 g + e of query j
        f32x4 sacc[TT];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) sacc[tt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        // (the block's tiles in turn, so that a matrix instruction does not
        // wait for the one before it)
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            half8 kf[TT];
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                const uint32_t rr = 16 * tt + j, piece = (4 * s + g) ^ (rr % T::kPieces);
                kf[tt] = *reinterpret_cast<const half8*>(cur.k + rr * (HD * 2) + 16 * piece);
            }
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) sacc[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[tt], qh[s], sacc[tt], 0, 0, 0);
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) sacc[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[tt], ql[s], sacc[tt], 0, 0, 0);
        }
        // Only the blocks past the tile's first query's position hold keys
        // that some of its queries don't see.
        const bool masked = kb * KB + KB > a.first + q0 + 1;
        float sc[TT][4];
        float bm = -__builtin_inff();
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float x = sacc[tt][e];
                if (cap) x = a.softcap * tanhf(fminf(fmaxf(x / a.softcap, -10.0f), 10.0f)) * kLog2e;
                sc[tt][e] = x;
            }
        if (masked) {
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (kb * KB + 16 * tt + 4 * g + e > qpos) sc[tt][e] = -__builtin_inff();
        }
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int e = 0; e < 4; ++e) bm = fmaxf(bm, sc[tt][e]);
        {
            const uint2 a16 = swap_rows<16>(__float_as_uint(bm));
            bm = fmaxf(__uint_as_float(a16.x), __uint_as_float(a16.y));
            const uint2 a32 = swap_rows<32>(__float_as_uint(bm));
            bm = fmaxf(__uint_as_float(a32.x), __uint_as_float(a32.y));
        }
        const float mn = fmaxf(m, bm);
        const float factor = __builtin_amdgcn_exp2f(m - mn);
        float bs = 0.0f;
        half8 ph[TT / 2], pl[TT / 2];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float p = __builtin_amdgcn_exp2f(sc[tt][e] - mn);
                bs += p;
                const _Float16 hi = static_cast<_Float16>(p);
                ph[tt / 2][4 * (tt % 2) + e] = hi;
                pl[tt / 2][4 * (tt % 2) + e] = static_cast<_Float16>(p - static_cast<float>(hi));
            }
        lsum = lsum * factor + bs;
        m = mn;
        // O^T: lane (j, g) gives V^T at dim 16 dt + j of keys 4 g .. 4 g + 3
        // and 16 + 4 g .. 16 + 4 g + 3 of each 32, the keys its P^T holds
        // (once the maxima have settled, most blocks leave the output's scale)
        if (__any(factor != 1.0f)) {
#pragma unroll
            for (int dt = 0; dt < HD / 16; ++dt)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[dt][e] *= factor;
        }
        constexpr int DT = KB == 64 ? 4 : 2;  // 16-dim tiles in turn, as the scores'
#pragma unroll
        for (int d0 = 0; d0 < HD / 16; d0 += DT)
#pragma unroll
            for (int u = 0; u < TT / 2; ++u) {
                half8 va[DT];
#pragma unroll
                for (int i = 0; i < DT; ++i) {
                    const _Float16* row = cur.vt + (16 * (d0 + i) + j) * T::kVtStride + 4 * g + 32 * u;
                    const uint2 lo = *reinterpret_cast<const uint2*>(row), hi = *reinterpret_cast<const uint2*>(row + 16);
                    va[i] = __builtin_bit_cast(half8, make_uint4(lo.x, lo.y, hi.x, hi.y));
                }
#pragma unroll
                for (int i = 0; i < DT; ++i) o[d0 + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[i], ph[u], o[d0 + i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < DT; ++i) o[d0 + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[i], pl[u], o[d0 + i], 0, 0, 0);
            }
    };
    for (uint32_t kb = 0; kb < blocks; kb += 2) {
        block(kb, s_t[0], s_t[1]);
        if (kb + 1 < blocks) block(kb + 1, s_t[1], s_t[0]);
    }
    // lane (j, g) holds dims 16 dt + 4 g .. + 3 of query j
    const uint2 l16 = swap_rows<16>(__float_as_uint(lsum));
    lsum = __uint_as_float(l16.x) + __uint_as_float(l16.y);
    const uint2 l32 = swap_rows<32>(__float_as_uint(lsum));
    lsum = __uint_as_float(l32.x) + __uint_as_float(l32.y);
    if (qlive) {
        const float inv = 1.0f / lsum;
        float* op = a.out + (static_cast<uint64_t>(qi) * a.heads + h) * HD + 4 * g;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt)
            *reinterpret_cast<float4*>(op + 16 * dt) = make_float4(o[dt][0] * inv, o[dt][1] * inv, o[dt][2] * inv, o[dt][3] * inv);
    }
}

const char* check_prompt(const vkml_attend_prompt_params* p) {
    if (!p) return "null params";
    if (p->kv_type != VKML_F16) return "caches must be f16";
    if (p->head_dim != 64 && p->head_dim != 128) return "head_dim must be 64 or 128";
    if (p->kv_heads == 0 || p->heads % p->kv_heads || (p->heads / p->kv_heads) % kHeads)
        return "query heads a KV head must be a multiple of 4";
    if (p->t == 0) return "no queries";
    if (static_cast<uint64_t>(p->first) + p->t > p->capacity) return "the keys do not fit the caches";
    return nullptr;
}

}  // namespace

extern "C" {

int vkml_attend_prompt_fast_supported(const vkml_attend_prompt_params* p) {
    return vkml::abi::initialized() && !check_prompt(p) ? 1 : 0;
}

int vkml_attend_prompt_fast(const vkml_attend_prompt_params* p, const float* q, const void* k_cache, const void* v_cache, float* out) {
    VKML_REQUIRE_INIT();
    if (const char* why = check_prompt(p)) return vkml::abi::fail(VKML_ERROR_INVALID_ARGUMENT, std::string("attend_prompt_fast: ") + why);
    VKML_CHECK_ARG(q && k_cache && v_cache && out, "attend_prompt_fast: null buffer");
    const PromptArgs a{q, k_cache, v_cache, out, p->heads, p->kv_heads, p->heads / p->kv_heads, p->capacity, p->t, p->first,
                       p->scale, p->softcap};
    const dim3 grid((p->t + kQueries - 1) / kQueries * (p->kv_heads * (a.group / kHeads)));
    vkml::abi::ProfileScope prof("attend_prompt_fast");
    const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, vkml::abi::stream(), a); };
    const bool wide = vkml::rules::wide_blocks(*p, grid.x, vkml::abi::compute_units());
    if (p->head_dim == 128) wide ? go(k_attend_prompt_fast<128, 64>) : go(k_attend_prompt_fast<128, 32>);
    else wide ? go(k_attend_prompt_fast<64, 64>) : go(k_attend_prompt_fast<64, 32>);
    return vkml::abi::check_launch("attend_prompt_fast");
}

}  // extern "C"
