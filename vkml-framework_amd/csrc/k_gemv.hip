// k_gemv.hip -- quantized matrix-vector products for decoding (the
// reference's shaders/gemv_dot.comp and gemv.comp), written for gfx950.
//
// The int8 path's device code (mapping, bit-exact order) is in gemv.hpp;
// here are its kernels, their launch shapes and the C ABI. 16 lanes a row
// are used when 8 would leave SIMDs idle (the N = 4096 projections of a 7B
// model: 4096 rows x 16 lanes is one wave per SIMD).
#include <algorithm>
#include <type_traits>

#include "device.hpp"
#include "gemv.hpp"
#include "internal.hpp"
#include "rules.hpp"

using namespace vkml::dev;
using namespace vkml::gemv;

namespace {

template <int FMT, bool F16S, int LPR, int EPI, int B, uint32_t T, int NORM, bool QOUT, bool FULL, int PRE = 1>
__global__ void __launch_bounds__(T) k_gemv_dot(GemvArgs g) {
    extern __shared__ uint4 smem[];
    GemvRows<FMT, F16S, LPR, EPI, B, T, QOUT, false, PRE, FULL> rows;
    if constexpr (PRE == 0) {
        // Every weight load of the row is issued at once: the activation's
        // loads go first, so that staging waits for them alone.
        StageLoads<T, NORM> act;
        stage_load<T, NORM, false>(g, act);
        rows.start(g, blockIdx.x);
        stage_store<T, NORM, false>(g, smem, act);
    } else if constexpr (NORM != 0) {
        // (the norm prologue's loads after the weights': measured faster)
        rows.start(g, blockIdx.x);  // the first batch of weights is in flight while the activation is staged
        stage_activation<T, NORM, false>(g, smem);
    } else {
        StageLoads<T, false> act;
        stage_load<T, false, false>(g, act);  // first: staging waits for these alone
        rows.start(g, blockIdx.x);            // the first batch of weights is in flight while the activation is staged
        stage_store<T, false, false>(g, smem, act);
    }
    rows.finish(g, smem, staged_ss(smem, g.k));
}

// Rows of up to 4096 values at 32 lanes a row: every round of the row is
// one batch, all in flight at once (T threads, T / 32 rows a workgroup).
template <int FMT, bool F16S, int EPI, int NORM, bool QOUT, uint32_t T>
int launch_deep(const GemvArgs& g, const char* label) {
    const dim3 grid((g.n + T / 32 - 1) / (T / 32));
    const size_t lds = stage_bytes(g.k, NORM != 0);
    if (g.k <= 2048) {
        if (g.k == 2048)
            hipLaunchKernelGGL((k_gemv_dot<FMT, F16S, 32, EPI, 4, T, NORM, QOUT, true, 0>), grid, dim3(T), lds, vkml::abi::stream(), g);
        else
            hipLaunchKernelGGL((k_gemv_dot<FMT, F16S, 32, EPI, 4, T, NORM, QOUT, false, 0>), grid, dim3(T), lds, vkml::abi::stream(), g);
    } else {
        if (g.k == 4096)
            hipLaunchKernelGGL((k_gemv_dot<FMT, F16S, 32, EPI, 8, T, NORM, QOUT, true, 0>), grid, dim3(T), lds, vkml::abi::stream(), g);
        else
            hipLaunchKernelGGL((k_gemv_dot<FMT, F16S, 32, EPI, 8, T, NORM, QOUT, false, 0>), grid, dim3(T), lds, vkml::abi::stream(), g);
    }
    return vkml::abi::check_launch(label);
}

// The batch pipeline (B rounds a batch, two batches in flight), T threads.
template <int FMT, bool F16S, int LPR, int EPI, int NORM, bool QOUT, uint32_t T>
int launch_batched(const GemvArgs& g, const char* label) {
    constexpr int B = LPR == 16 ? 4 : 2;  // rounds per batch (2 measured best at 32 lanes)
    const dim3 grid((g.n + T / LPR - 1) / (T / LPR));
    const size_t lds = stage_bytes(g.k, NORM != 0);
    // Whole pairs of whole batches (K a multiple of 1024 B) need no per-lane
    // tail check and no per-round test (q4_K and q8_0 kernels are built both
    // ways).
    constexpr bool kWhole = FMT == VKML_Q4_K || FMT == VKML_Q8_0;
    if (kWhole && g.k % (1024 * B) == 0)
        hipLaunchKernelGGL((k_gemv_dot<FMT, F16S, LPR, EPI, B, T, NORM, QOUT, kWhole>), grid, dim3(T), lds, vkml::abi::stream(), g);
    else
        hipLaunchKernelGGL((k_gemv_dot<FMT, F16S, LPR, EPI, B, T, NORM, QOUT, false>), grid, dim3(T), lds, vkml::abi::stream(), g);
    return vkml::abi::check_launch(label);
}

template <int FMT, bool F16S, int LPR, int EPI, int NORM, bool QOUT>
int launch(const GemvArgs& g, const char* label) {
    // (512 threads with the norm prologue at 32 lanes: half the workgroups
    // redo RMSNorm + Q8_0 of x, each over twice the threads)
    constexpr uint32_t T = QOUT ? 32 * LPR : LPR == 32 ? (NORM != 0 ? 512 : 256) : 128;
    vkml::abi::ProfileScope prof(label);
    const uint32_t cus = vkml::abi::compute_units();
    constexpr bool kWhole = FMT == VKML_Q4_K || FMT == VKML_Q8_0;
    if constexpr (kWhole && LPR == 32) {
        if (g.k <= 4096) {
            // With the norm prologue, which every workgroup computes over the
            // whole row: 24 rows a workgroup where that makes one workgroup a
            // compute unit (the N = 6144 q|k|v projection of a 7B model).
            if constexpr (NORM != 0) {
                if ((g.n + 15) / 16 > cus && (g.n + 23) / 24 <= cus) {
                    // q4_K rows of 4096 with the store epilogue (a decode
                    // step's q|k|v): 16 lanes a row over 384 threads, the
                    // same 24 rows a workgroup. 32 lanes load each 16-byte
                    // code group twice (lanes l and l ^ 2), 16 lanes once, so
                    // a compute unit queues half the code loads (measured:
                    // 606.6 against 605.3 tokens/s at cfg5).
                    if constexpr (FMT == VKML_Q4_K && EPI == kStore) {
                        if (g.k == 4096) {
                            hipLaunchKernelGGL((k_gemv_dot<FMT, F16S, 16, EPI, 8, 384, NORM, QOUT, true, 0>), dim3((g.n + 23) / 24),
                                               dim3(384), stage_bytes(g.k, true), vkml::abi::stream(), g);
                            return vkml::abi::check_launch(label);
                        }
                    }
                    return launch_deep<FMT, F16S, EPI, NORM, QOUT, 768>(g, label);
                }
            }
            return launch_deep<FMT, F16S, EPI, NORM, QOUT, T>(g, label);
        }
    }
    return launch_batched<FMT, F16S, LPR, EPI, NORM, QOUT, T>(g, label);
}

template <int FMT, bool F16S, int EPI, int NORM, bool QOUT>
int dispatch(const GemvArgs& g, const char* label) {
    // 8 lanes a row unless that leaves fewer than one wave per SIMD; 32
    // (q4_K, q8_0) when 16 would leave fewer than two, so that one wave's
    // arithmetic overlaps another's loads (the N = 4096 and 6144 projections
    // of a 7B model: measured 13-18% faster than 16 lanes).
    const uint64_t simds = 4ull * std::max<uint32_t>(vkml::abi::compute_units(), 1);
    if constexpr (FMT == VKML_Q4_K || FMT == VKML_Q8_0) {
        // (their buffer loads address a matrix under 4 GiB)
        if (code_bytes<FMT>(g.n, g.k) >= (1ull << 32) || scale_bytes<FMT, F16S>(g.n, g.k) >= (1ull << 32))
            return vkml::abi::fail(VKML_ERROR_UNSUPPORTED, std::string(label) + ": a matrix of 4 GiB or more");
        if constexpr (!QOUT) {
            if ((g.n + 3) / 4 < 2 * simds) return launch<FMT, F16S, 32, EPI, NORM, QOUT>(g, label);
        }
    }
    if ((g.n + 7) / 8 < simds) return launch<FMT, F16S, 16, EPI, NORM, QOUT>(g, label);
    return launch<FMT, F16S, 8, EPI, NORM, QOUT>(g, label);
}

template <int EPI, int NORM = 0, bool QOUT = false>
int dispatch_format(uint32_t b_type, uint32_t scale_type, const GemvArgs& g, const char* label) {
    const bool f16 = scale_type == VKML_F16;
    switch (b_type) {
        case VKML_Q8_0: return f16 ? dispatch<VKML_Q8_0, true, EPI, NORM, QOUT>(g, label) : dispatch<VKML_Q8_0, false, EPI, NORM, QOUT>(g, label);
        case VKML_Q4_0: return f16 ? dispatch<VKML_Q4_0, true, EPI, NORM, QOUT>(g, label) : dispatch<VKML_Q4_0, false, EPI, NORM, QOUT>(g, label);
        case VKML_Q4_1: return f16 ? dispatch<VKML_Q4_1, true, EPI, NORM, QOUT>(g, label) : dispatch<VKML_Q4_1, false, EPI, NORM, QOUT>(g, label);
        case VKML_Q4_K: return dispatch<VKML_Q4_K, true, EPI, NORM, QOUT>(g, label);
        default: return vkml::abi::fail(VKML_ERROR_UNSUPPORTED, std::string(label) + ": no int8 kernel for weight type " + std::to_string(b_type));
    }
}

int check_dot_params(const vkml_gemv_dot_params* p, const char* what, bool any_k = false) {
    VKML_REQUIRE_INIT();
    VKML_CHECK_ARG(p, std::string(what) + ": null params");
    VKML_CHECK_ARG(p->b_type == VKML_Q8_0 || p->b_type == VKML_Q4_0 || p->b_type == VKML_Q4_1 || p->b_type == VKML_Q4_K,
                   std::string(what) + ": weights must be q8_0, q4_0, q4_1 or q4_K, got type " + std::to_string(p->b_type));
    VKML_CHECK_ARG(p->b_type == VKML_Q4_K || p->scale_type == VKML_F16 || p->scale_type == VKML_F32,
                   std::string(what) + ": scales must be f16 or f32");
    const uint32_t unit = p->b_type == VKML_Q4_K ? 256 : 32;
    VKML_CHECK_ARG(p->k > 0 && p->k % unit == 0 && (any_k || p->k <= kMaxK),
                   std::string(what) + ": k = " + std::to_string(p->k) + " must be a positive multiple of " +
                       std::to_string(unit) + (any_k ? std::string() : " up to " + std::to_string(kMaxK)));
    return VKML_OK;
}

// ---------------------------------------------------------------- several rows

// gemv_dot for 2 .. 8 activation rows in one launch (gemv_dot.comp handles
// its M rows in one dispatch): each round of a weight row is loaded and
// unpacked once and applied to every activation row, each row with its own
// accumulators in the single-row kernel's order (the same lanes, terms and
// halving tree). LPR lanes an output row. K runs in chunks of CR rounds (four,
// fewer for short rows): the workgroup stages the chunk's codes, code sums and scales of every
// activation row in LDS, and the next chunk's weights and activations are in
// flight meanwhile. At two rows bound by reading the weights; each further
// row adds ten VALU operations and 24 bytes from LDS a half-block and lane,
// which bound it from four on. Against reading the activations from the
// caches and summing their codes a lane (us; two, five and eight rows):
// q4_K 14336 x 4096 17.6, 24.5, 32.3 -> 11.4, 17.7, 20.7; 4096 x 14336 23.1,
// 28.9, 35.0 -> 11.5, 17.7, 21.0; q8_0 4096 x 14336 22.5, 26.4, 31.1 -> 12.2,
// 16.5, 19.2; q4_0 14336 x 4096 12.7, 21.9, 30.1 -> 10.0, 16.3, 19.5. (Two
// weight rows a lane sharing the LDS reads: within 5% either way.)
template <int FMT, bool F16S, int LPR, bool FULL, int M, uint32_t CR>
__global__ void __launch_bounds__(256) k_gemv_dot_rows(GemvArgs g, uint32_t m) {
    constexpr int NS = Plan<FMT, LPR>::NS;
    constexpr uint32_t kRows = 256 / LPR, H = 32 * CR, NL = (M * H + 255) / 256;
    __shared__ uint4 s_codes[M][H];
    __shared__ float2 s_ss[M][H];
    const uint32_t t = thread_index(), l = t % LPR, grp = t / LPR;
    const uint32_t out_row = blockIdx.x * kRows + grp, row = min(out_row, g.n - 1);
    const uint32_t K = g.k, halves = K / 16, rounds = (halves + 31) / 32;
    const Q4kField jf = q4k_field((l % 16) / 2);
    // Rows past m repeat the last one and are not stored; half-blocks past K
    // repeat its last one and are skipped.
    uint4 codes[NL];
    float scale[NL];
    const auto load_act = [&](uint32_t r0) {
#pragma unroll
        for (uint32_t u = 0; u < NL; ++u) {
            const uint32_t e = t + 256 * u, i = min(e / H, m - 1), hb = min(32 * r0 + e % H, halves - 1);
            if (M * H % 256 != 0 && e >= M * H) break;
            codes[u] = ldg(g.a_values + static_cast<uint64_t>(i) * halves + hb);
            scale[u] = ldg(g.a_scales + static_cast<uint64_t>(i) * (K / 32) + hb / 2);
        }
    };
    RoundW<FMT, LPR> w[CR], next[CR];
    const auto load_weights = [&](uint32_t r0, RoundW<FMT, LPR> (&d)[CR]) {
#pragma unroll
        for (uint32_t u = 0; u < CR; ++u) load_round<FMT, F16S, LPR>(g.b_values, g.b_scales, K, row, min(r0 + u, rounds - 1), l, d[u]);
    };
    float acc[M][NS];
#pragma unroll
    for (int i = 0; i < M; ++i)
#pragma unroll
        for (int e = 0; e < NS; ++e) acc[i][e] = 0.0f;
    load_act(0);
    load_weights(0, w);
    for (uint32_t r0 = 0; r0 < rounds; r0 += CR) {
        __syncthreads();  // the last chunk's readers are done
#pragma unroll
        for (uint32_t u = 0; u < NL; ++u) {
            const uint32_t e = t + 256 * u;
            if (M * H % 256 != 0 && e >= M * H) break;
            s_codes[e / H][e % H] = codes[u];
            s_ss[e / H][e % H] = make_float2(static_cast<float>(byte_sum(codes[u])), scale[u]);
        }
        __syncthreads();
        if (r0 + CR < rounds) {
            load_act(r0 + CR);
            load_weights(r0 + CR, next);
        }
        // Two activation rows at a time, the next two's LDS reads issued before
        // this two's arithmetic (left to itself the compiler waits for each
        // read where it issues it).
        RoundA<FMT, LPR> x[2][2];
        const auto fetch = [&](uint32_t u, uint32_t i, RoundA<FMT, LPR>& d) {
#pragma unroll
            for (int e = 0; e < NS; ++e) {
                const uint32_t hb = 32 * u + acc_index<FMT, LPR>(l, e);
                d.a[e] = s_codes[i][hb];
                d.ss[e] = s_ss[i][hb];
            }
        };
        fetch(0, 0, x[0][0]);
        fetch(0, 1, x[0][1]);
#pragma unroll
        for (uint32_t u = 0; u < CR; ++u) {
            if (r0 + u >= rounds) break;
#pragma unroll
            for (uint32_t i = 0; i < M; i += 2) {
                const uint32_t p = (u * (M / 2) + i / 2) % 2;
                if (i + 2 < M || u + 1 < CR) {
                    const uint32_t nu = i + 2 < M ? u : u + 1, ni = i + 2 < M ? i + 2 : 0;
                    fetch(nu, ni, x[1 - p][0]);
                    fetch(nu, ni + 1, x[1 - p][1]);
                }
                __builtin_amdgcn_sched_barrier(0);
                round_terms<FMT, F16S, LPR, FULL>(w[u], x[p][0], r0 + u, l, K, jf, acc[i]);
                round_terms<FMT, F16S, LPR, FULL>(w[u], x[p][1], r0 + u, l, K, jf, acc[i + 1]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < CR; ++u) w[u] = next[u];
    }
#pragma unroll
    for (int i = 0; i < M; ++i) {
        if (i >= static_cast<int>(m)) break;
        const float v = row_tree<FMT, LPR>(acc[i]);
        // + residual (one activation row): add(x, y), llama.cpp:374,386
        if (l == 0 && out_row < g.n) g.out[static_cast<uint64_t>(i) * g.n + out_row] = g.residual ? ldg(g.residual + out_row) + v : v;
    }
}

template <int FMT, bool F16S>
int launch_rows(const GemvArgs& g, uint32_t m) {
    // 32 lanes a row where the format has them (16 lanes, half the waves and
    // twice the accumulators a lane: 24.5 against 18.1 us at 14336 x 4096,
    // q4_K, five rows).
    constexpr int LPR = FMT == VKML_Q8_0 || FMT == VKML_Q4_K ? 32 : 16;
    const dim3 grid((g.n + 256 / LPR - 1) / (256 / LPR));
    vkml::abi::ProfileScope prof("gemv_dot");
    const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, vkml::abi::stream(), g, m); };
    const auto chunk = [&](auto cr) {
        constexpr uint32_t CR = decltype(cr)::value;
        const bool full = g.k % 512 == 0;
        if (m <= 2) full ? go(k_gemv_dot_rows<FMT, F16S, LPR, true, 2, CR>) : go(k_gemv_dot_rows<FMT, F16S, LPR, false, 2, CR>);
        else if (m <= 4) full ? go(k_gemv_dot_rows<FMT, F16S, LPR, true, 4, CR>) : go(k_gemv_dot_rows<FMT, F16S, LPR, false, 4, CR>);
        else if (m <= 6) full ? go(k_gemv_dot_rows<FMT, F16S, LPR, true, 6, CR>) : go(k_gemv_dot_rows<FMT, F16S, LPR, false, 6, CR>);
        else full ? go(k_gemv_dot_rows<FMT, F16S, LPR, true, 8, CR>) : go(k_gemv_dot_rows<FMT, F16S, LPR, false, 8, CR>);
    };
    switch (vkml::rules::rows_chunk(g.k)) {
        case 1: chunk(std::integral_constant<uint32_t, 1>()); break;
        case 2: chunk(std::integral_constant<uint32_t, 2>()); break;
        default: chunk(std::integral_constant<uint32_t, 4>()); break;
    }
    return vkml::abi::check_launch("gemv_dot");
}

int dispatch_rows(uint32_t fmt, uint32_t st, const GemvArgs& g, uint32_t m) {
    const bool f16 = st == VKML_F16;
    switch (fmt) {
        case VKML_Q8_0: return f16 ? launch_rows<VKML_Q8_0, true>(g, m) : launch_rows<VKML_Q8_0, false>(g, m);
        case VKML_Q4_0: return f16 ? launch_rows<VKML_Q4_0, true>(g, m) : launch_rows<VKML_Q4_0, false>(g, m);
        case VKML_Q4_1: return f16 ? launch_rows<VKML_Q4_1, true>(g, m) : launch_rows<VKML_Q4_1, false>(g, m);
        default: return launch_rows<VKML_Q4_K, true>(g, m);
    }
}

// ---------------------------------------------------------------- float path

// gemv.comp's order: 32 lanes per output, lane l taking the 4-element
// groups l, l + 32, ... of its row (dot(a4, w) summed left to right), then
// the halving tree over the 32 lanes (gemv.comp:117-212). Two rows a wave.
// Batch blockIdx.y multiplies its a by float b's batch y / b_group.
template <int BT>
__global__ void __launch_bounds__(256) k_gemv_float(const float* a, uint32_t m, const void* b, const void* bs, uint32_t st,
                                                    float* out, uint32_t n, uint32_t k, uint32_t b_group, uint64_t b_stride) {
#pragma clang fp contract(off)
    const uint32_t z = blockIdx.y;
    a += static_cast<uint64_t>(z) * m * k;
    out += static_cast<uint64_t>(z) * m * n;
    if constexpr (BT <= VKML_BF16) {
        const uint64_t off = static_cast<uint64_t>(z / b_group) * b_stride * (BT == VKML_F32 ? 4 : 2);
        b = static_cast<const uint8_t*>(b) + off;
    }
    const uint32_t lane = threadIdx.x % 32;
    const uint32_t row = blockIdx.x * (blockDim.x / 32) + threadIdx.x / 32;
    const uint32_t r = min(row, n - 1);
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    const auto w_at = [&](uint64_t col) -> float {
        if constexpr (BT == VKML_F32) return static_cast<const float*>(b)[static_cast<uint64_t>(r) * k + col];
        else return weight_value(BT, st, b, bs, k, r, col);
    };
    if (k % 4 == 0) {
        for (uint32_t i = lane; i < k / 4; i += 32) {
            const float w0 = w_at(4 * i), w1 = w_at(4 * i + 1), w2 = w_at(4 * i + 2), w3 = w_at(4 * i + 3);
#pragma unroll
            for (uint32_t q = 0; q < 8; ++q) {
                if (q < m) {
                    const float* ar = a + static_cast<uint64_t>(q) * k + 4 * i;
                    acc[q] += ar[0] * w0 + ar[1] * w1 + ar[2] * w2 + ar[3] * w3;
                }
            }
        }
    } else {
        for (uint32_t col = lane; col < k; col += 32) {
            const float w = w_at(col);
#pragma unroll
            for (uint32_t q = 0; q < 8; ++q)
                if (q < m) acc[q] += a[static_cast<uint64_t>(q) * k + col] * w;
        }
    }
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) {
        if (q >= m) break;
        const float v = tree_to_first<32>(acc[q]);  // strides 16 .. 1 toward the row's lane 0
        if (lane == 0 && row < n) out[static_cast<uint64_t>(q) * n + row] = v;
    }
}

// The same order for a float b whose rows are whole, aligned groups of four
// (k % 4 == 0): a lane loads a group with one 8- or 16-byte load, U steps of
// R rows at once, the next batch's loads in flight while this one is summed,
// a from the caches. For rows of one or two steps (scores of 32 heads of 128
// against 4000 keys: two queries 20 -> 11 us, eight 30 -> 23.5; a row a half
// wave where the outputs are few, two rows of a by 1000 x 64 2.4 -> 2.1), and
// for one row of a by an f32 b past the last-level cache (gemv_row_cached).
template <int BT>
using Group4 = std::conditional_t<BT == VKML_F32, uint4, uint2>;

template <int BT>
__device__ __forceinline__ float4 widen4(Group4<BT> w) {
    if constexpr (BT == VKML_F32) return make_float4(__uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w));
    else return make_float4(half_to_float(w.x & 0xFFFFu, BT), half_to_float(w.x >> 16, BT), half_to_float(w.y & 0xFFFFu, BT),
                            half_to_float(w.y >> 16, BT));
}

template <int BT, int M, int R, int U>
__global__ void __launch_bounds__(256) k_gemv_float4(const float* a, uint32_t m, const void* b, float* out, uint32_t n, uint32_t k,
                                                     uint32_t b_group, uint64_t b_stride) {
#pragma clang fp contract(off)
    constexpr uint32_t kSize = BT == VKML_F32 ? 4 : 2;
    const uint32_t z = blockIdx.y, lane = threadIdx.x % 32, groups = k / 4;
    a += static_cast<uint64_t>(z) * m * k;
    out += static_cast<uint64_t>(z) * m * n;
    const uint8_t* bz = static_cast<const uint8_t*>(b) + static_cast<uint64_t>(z / b_group) * b_stride * kSize;
    const uint32_t row0 = (blockIdx.x * 8 + threadIdx.x / 32) * R;
    const Group4<BT>* br[R];
#pragma unroll
    for (int r = 0; r < R; ++r) br[r] = reinterpret_cast<const Group4<BT>*>(bz + static_cast<uint64_t>(min(row0 + r, n - 1)) * k * kSize);
    const float4* ar[M];  // (rows past m repeat the last one, and are not stored)
#pragma unroll
    for (int q = 0; q < M; ++q) ar[q] = reinterpret_cast<const float4*>(a + static_cast<uint64_t>(min(static_cast<uint32_t>(q), m - 1)) * k);
    struct Batch {
        Group4<BT> w[U][R];
        float4 x[U][M];
    };
    const auto load = [&](uint32_t s, Batch& d) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t i = min(32 * (s + u) + lane, groups - 1);
#pragma unroll
            for (int r = 0; r < R; ++r) d.w[u][r] = ldg(br[r] + i);
#pragma unroll
            for (int q = 0; q < M; ++q) d.x[u][q] = ldg(ar[q] + i);
        }
    };
    float acc[M][R];
#pragma unroll
    for (int q = 0; q < M; ++q)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[q][r] = 0.0f;
    const auto step = [&](uint32_t u, const Batch& d) {
        float4 w[R];
#pragma unroll
        for (int r = 0; r < R; ++r) w[r] = widen4<BT>(d.w[u][r]);
#pragma unroll
        for (int q = 0; q < M; ++q) {
            const float4 x = d.x[u][q];
#pragma unroll
            for (int r = 0; r < R; ++r) acc[q][r] += x.x * w[r].x + x.y * w[r].y + x.z * w[r].z + x.w * w[r].w;
        }
    };
    const uint32_t steps = (groups + 31) / 32;
    Batch cur, next;
    load(0, cur);
    for (uint32_t s = 0; s < steps; s += U) {
        if (s + U < steps) load(s + U, next);
        if (32 * (s + U) <= groups) {
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) step(u, cur);
        } else {
#pragma unroll
            for (uint32_t u = 0; u < U; ++u)
                if (32 * (s + u) + lane < groups) step(u, cur);
        }
        cur = next;
    }
#pragma unroll
    for (int q = 0; q < M; ++q) {
        if (q >= static_cast<int>(m)) break;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float v = tree_to_first<32>(acc[q][r]);  // strides 16 .. 1 toward the row's lane 0
            if (lane == 0 && row0 + r < n) out[static_cast<uint64_t>(q) * n + row0 + r] = v;
        }
    }
}

// The same for longer rows: a's groups, which every row of b needs, are
// staged in LDS, eight steps (1024 values of each row of a) at a time, the
// next chunk's loads of a and of b in flight meanwhile. Bound by reading b
// (one row of b a half wave, us against the kernel above it, which loads an
// element at a time and waits for each group): bf16 14336 x 4096, one row of
// a 39.8 -> 23.4 (5.0 TB/s), five 77.3 -> 34.5, eight 107 -> 45; 4096 x
// 14336 84.1 -> 24.2, 198 -> 46.6, 281 -> 56; two rows of b a half wave lose
// at n = 4096 (51.5 against 37 at four rows of a). From six rows of a on, the
// products and sums, two VALU operations each, weigh as much as b.
template <int BT, int M>
__global__ void __launch_bounds__(256) k_gemv_float4_rows(const float* a, uint32_t m, const void* b, float* out, uint32_t n, uint32_t k,
                                                          uint32_t b_group, uint64_t b_stride) {
#pragma clang fp contract(off)
    constexpr uint32_t kSize = BT == VKML_F32 ? 4 : 2;
    constexpr uint32_t U = 8;
    __shared__ float4 xs[M][32 * U];
    const uint32_t z = blockIdx.y, t = threadIdx.x, lane = t % 32, groups = k / 4;
    a += static_cast<uint64_t>(z) * m * k;
    out += static_cast<uint64_t>(z) * m * n;
    const uint8_t* bz = static_cast<const uint8_t*>(b) + static_cast<uint64_t>(z / b_group) * b_stride * kSize;
    const uint32_t row = blockIdx.x * 8 + t / 32;
    const Group4<BT>* br = reinterpret_cast<const Group4<BT>*>(bz + static_cast<uint64_t>(min(row, n - 1)) * k * kSize);
    const float4* a4 = reinterpret_cast<const float4*>(a);
    float4 xa[M];  // group t of the chunk, of every row of a (rows past m repeat the last one, and are not stored)
    Group4<BT> cur[U], next[U];
    const auto load = [&](uint32_t s, Group4<BT> (&w)[U]) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) w[u] = ldg(br + min(32 * (s + u) + lane, groups - 1));
#pragma unroll
        for (int q = 0; q < M; ++q) xa[q] = ldg(a4 + static_cast<uint64_t>(min(static_cast<uint32_t>(q), m - 1)) * groups + min(32 * s + t, groups - 1));
    };
    float acc[M];
#pragma unroll
    for (int q = 0; q < M; ++q) acc[q] = 0.0f;
    const uint32_t steps = (groups + 31) / 32;
    load(0, cur);
    for (uint32_t s = 0; s < steps; s += U) {
        __syncthreads();  // the last chunk's readers are done
#pragma unroll
        for (int q = 0; q < M; ++q) xs[q][t] = xa[q];
        __syncthreads();
        if (s + U < steps) load(s + U, next);
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            if (32 * (s + u) + lane < groups) {
                const float4 w = widen4<BT>(cur[u]);
#pragma unroll
                for (int q = 0; q < M; ++q) {
                    const float4 x = xs[q][32 * u + lane];
                    acc[q] += x.x * w.x + x.y * w.y + x.z * w.z + x.w * w.w;
                }
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) cur[u] = next[u];
    }
#pragma unroll
    for (int q = 0; q < M; ++q) {
        if (q >= static_cast<int>(m)) break;
        const float v = tree_to_first<32>(acc[q]);  // strides 16 .. 1 toward the row's lane 0
        if (lane == 0 && row < n) out[static_cast<uint64_t>(q) * n + row] = v;
    }
}

// One row of b a half wave, its U steps at once.
template <int BT, int U, class Go>
void short_rows(const Go& go, uint32_t m) {
    if (m == 1) go(k_gemv_float4<BT, 1, 1, U>, 1);
    else if (m == 2) go(k_gemv_float4<BT, 2, 1, U>, 1);
    else if (m <= 4) go(k_gemv_float4<BT, 4, 1, U>, 1);
    else if (m <= 6) go(k_gemv_float4<BT, 6, 1, U>, 1);
    else go(k_gemv_float4<BT, 8, 1, U>, 1);
}

template <int BT>
void launch_float4(const vkml_gemv_params& p, const float* a, const void* b, float* out, uint32_t batches, uint32_t group) {
    const auto go = [&](auto kernel, uint32_t rows) {
        hipLaunchKernelGGL(kernel, dim3((p.n + 8 * rows - 1) / (8 * rows), batches), dim3(256), 0, vkml::abi::stream(), a, p.m, b, out, p.n, p.k,
                           group, static_cast<uint64_t>(p.b_stride));
    };
    if (p.k <= 256 && vkml::rules::gemv_row_each(p.m, p.n, batches)) {
        p.k <= 128 ? short_rows<BT, 1>(go, p.m) : short_rows<BT, 2>(go, p.m);
    } else if (p.k <= 256) {
        // One or two steps a row (attention's scores of up to 8 queries):
        // several rows a lane keep as many loads in flight, and a is read
        // from the caches.
        if (p.m == 1) go(k_gemv_float4<BT, 1, 4, 2>, 4);
        else if (p.m == 2) go(k_gemv_float4<BT, 2, 4, 2>, 4);
        else if (p.m <= 4) go(k_gemv_float4<BT, 4, 2, 1>, 2);
        else if (p.m <= 6) go(k_gemv_float4<BT, 6, 2, 1>, 2);
        else go(k_gemv_float4<BT, 8, 2, 1>, 2);
    } else if (vkml::rules::gemv_row_cached(p)) {
        if constexpr (BT == VKML_F32) go(k_gemv_float4<BT, 1, 1, 8>, 1);  // a from the caches
    } else if (p.m == 1) go(k_gemv_float4_rows<BT, 1>, 1);
    else if (p.m == 2) go(k_gemv_float4_rows<BT, 2>, 1);
    else if (p.m <= 4) go(k_gemv_float4_rows<BT, 4>, 1);
    else if (p.m <= 6) go(k_gemv_float4_rows<BT, 6>, 1);
    else go(k_gemv_float4_rows<BT, 8>, 1);
}

}  // namespace

extern "C" {

int vkml_gemv_dot(const vkml_gemv_dot_params* p, const void* a_values, const void* b_values, float* out,
                  const void* b_scales, const float* a_scales) {
    if (int r = check_dot_params(p, "gemv_dot", true)) return r;
    VKML_CHECK_ARG(p->m >= 1 && p->m <= 8, "gemv_dot: m must be 1 to 8, got " + std::to_string(p->m));
    if (p->n == 0) return VKML_OK;
    VKML_CHECK_ARG(a_values && b_values && out && b_scales && a_scales, "gemv_dot: null buffer");
    if (p->m > 1 || p->k > kMaxK) {
        const GemvArgs g{static_cast<const uint4*>(a_values), a_scales, b_values, b_scales, nullptr, nullptr, out, nullptr, p->n, p->k};
        return dispatch_rows(p->b_type, p->scale_type, g, p->m);
    }
    const GemvArgs g{static_cast<const uint4*>(a_values), a_scales, b_values, b_scales, nullptr, nullptr, out, nullptr, p->n, p->k};
    return dispatch_format<kStore>(p->b_type, p->scale_type, g, "gemv_dot");
}

int vkml_gemv_dot_add(const vkml_gemv_dot_params* p, const void* a_values, const void* b_values, float* out,
                      const void* b_scales, const float* a_scales, const float* residual) {
    if (int r = check_dot_params(p, "gemv_dot_add", true)) return r;
    VKML_CHECK_ARG(p->m == 1, "gemv_dot_add: m must be 1");
    if (p->n == 0) return VKML_OK;
    VKML_CHECK_ARG(a_values && b_values && out && b_scales && a_scales && residual, "gemv_dot_add: null buffer");
    GemvArgs g{static_cast<const uint4*>(a_values), a_scales, b_values, b_scales, nullptr, nullptr, out, residual, p->n, p->k};
    if (p->k > kMaxK) return dispatch_rows(p->b_type, p->scale_type, g, 1);  // the activation staged in chunks
    return dispatch_format<kAdd>(p->b_type, p->scale_type, g, "gemv_dot_add");
}

int vkml_gemv_dot_swiglu(const vkml_gemv_dot_params* p, const void* a_values, const float* a_scales,
                         const void* gate_values, const void* gate_scales, const void* up_values,
                         const void* up_scales, float* h) {
    if (int r = check_dot_params(p, "gemv_dot_swiglu")) return r;
    VKML_CHECK_ARG(p->m == 1, "gemv_dot_swiglu: m must be 1");
    if (p->n == 0) return VKML_OK;
    VKML_CHECK_ARG(a_values && a_scales && gate_values && gate_scales && up_values && up_scales && h,
                   "gemv_dot_swiglu: null buffer");
    GemvArgs g{static_cast<const uint4*>(a_values), a_scales, gate_values, gate_scales, up_values, up_scales, h, nullptr, p->n, p->k};
    return dispatch_format<kSwiglu>(p->b_type, p->scale_type, g, "gemv_dot_swiglu");
}

int vkml_gemv_fused(const vkml_gemv_fused_params* p, const void* a, const float* a_scales, const float* norm_weight,
                    const void* b_values, const void* b_scales, const void* b2_values, const void* b2_scales,
                    const float* residual, float* out, void* out_values, float* out_scales) {
    VKML_REQUIRE_INIT();
    VKML_CHECK_ARG(p, "gemv_fused: null params");
    const vkml_gemv_dot_params dp{1, p->n, p->k, p->b_type, p->scale_type};
    if (int r = check_dot_params(&dp, "gemv_fused")) return r;
    VKML_CHECK_ARG(p->epilogue <= 2, "gemv_fused: epilogue must be 0 (store), 1 (+ residual) or 2 (SwiGLU)");
    VKML_CHECK_ARG(!p->quantize_out || p->epilogue == 2, "gemv_fused: quantize_out needs the SwiGLU epilogue");
    VKML_CHECK_ARG(!p->quantize_out || p->n % 32 == 0, "gemv_fused: quantize_out needs n a multiple of 32");
    VKML_CHECK_ARG(p->norm <= 2, "gemv_fused: norm must be 0 (quantized input), 1 (RMSNorm + Q8_0) or 2 (Q8_0)");
    VKML_CHECK_ARG(!p->norm || p->k <= 4096, "gemv_fused: the RMSNorm / Q8_0 prologue takes k up to 4096");
    VKML_CHECK_ARG(!(p->norm && p->epilogue == 1), "gemv_fused: the RMSNorm / Q8_0 prologue goes with the store or SwiGLU epilogue");
    VKML_CHECK_ARG(p->norm != 2 || p->epilogue == 0, "gemv_fused: the plain Q8_0 prologue (norm 2) goes with the store epilogue");
    if (p->n == 0) return VKML_OK;
    VKML_CHECK_ARG(a && b_values && b_scales && out, "gemv_fused: null buffer");
    VKML_CHECK_ARG(p->norm == 1 ? norm_weight != nullptr : p->norm == 2 || a_scales != nullptr,
                   "gemv_fused: the input needs its norm weight or scales");
    VKML_CHECK_ARG(p->epilogue != 1 || residual, "gemv_fused: the residual epilogue needs the residual");
    VKML_CHECK_ARG(p->epilogue != 2 || (b2_values && b2_scales), "gemv_fused: SwiGLU needs the up matrix");
    VKML_CHECK_ARG(!p->quantize_out || (out_values && out_scales), "gemv_fused: quantize_out needs its buffers");
    GemvArgs g{p->norm ? nullptr : static_cast<const uint4*>(a), a_scales, b_values, b_scales, b2_values, b2_scales, out, residual,
               p->n, p->k, p->norm ? static_cast<const float*>(a) : nullptr, p->norm == 1 ? norm_weight : nullptr, p->eps,
               static_cast<uint8_t*>(out_values), out_scales};
    const char* label = "gemv_fused";
    switch (p->epilogue) {
        case 0: return p->norm == 1 ? dispatch_format<kStore, 1>(p->b_type, p->scale_type, g, label)
                       : p->norm == 2 ? dispatch_format<kStore, 2>(p->b_type, p->scale_type, g, label)
                                      : dispatch_format<kStore>(p->b_type, p->scale_type, g, label);
        case 1: return dispatch_format<kAdd>(p->b_type, p->scale_type, g, label);
        default:
            if (p->norm) {
                return p->quantize_out ? dispatch_format<kSwiglu, true, true>(p->b_type, p->scale_type, g, label)
                                       : dispatch_format<kSwiglu, true, false>(p->b_type, p->scale_type, g, label);
            }
            return p->quantize_out ? dispatch_format<kSwiglu, false, true>(p->b_type, p->scale_type, g, label)
                                   : dispatch_format<kSwiglu>(p->b_type, p->scale_type, g, label);
    }
}

int vkml_gemv_rope(const vkml_gemv_rope_params* p, const float* x, const float* norm_weight, const void* b_values,
                   const void* b_scales, float* qkv, const float* rope_table, const vkml_decode_state* state, void* k_cache,
                   void* v_cache) {
    VKML_REQUIRE_INIT();
    VKML_CHECK_ARG(p, "gemv_rope: null params");
    const vkml_gemv_dot_params dp{1, p->n, p->k, p->b_type, p->scale_type};
    if (int r = check_dot_params(&dp, "gemv_rope")) return r;
    VKML_CHECK_ARG(p->k <= 4096, "gemv_rope: the RMSNorm + Q8_0 prologue takes k up to 4096");
    VKML_CHECK_ARG(p->head_dim > 0 && p->head_dim % 2 == 0 && p->heads > 0 && p->kv_heads > 0 && p->capacity > 0,
                   "gemv_rope: heads, kv_heads, capacity and an even head_dim must be positive");
    VKML_CHECK_ARG(p->kv_type == VKML_F16 || p->kv_type == VKML_F32, "gemv_rope: caches must be f16 or f32");
    const uint64_t q_rows = static_cast<uint64_t>(p->heads) * p->head_dim, kv_rows = static_cast<uint64_t>(p->kv_heads) * p->head_dim;
    // Pairs of rows share a workgroup when the first row is even.
    VKML_CHECK_ARG(p->row0 % 2 == 0 && p->n % 2 == 0 && p->row0 + static_cast<uint64_t>(p->n) <= q_rows + 2 * kv_rows,
                   "gemv_rope: rows " + std::to_string(p->row0) + " .. " + std::to_string(p->row0 + p->n) + " must be even-aligned rows of the " +
                       std::to_string(q_rows + 2 * kv_rows) + " of [q | k | v]");
    if (p->n == 0) return VKML_OK;
    VKML_CHECK_ARG(x && norm_weight && b_values && b_scales && qkv && state && k_cache && v_cache && (rope_table || !p->rotate),
                   "gemv_rope: null buffer");
    GemvArgs g{nullptr, nullptr, b_values, b_scales, nullptr, nullptr, qkv + p->row0, nullptr, p->n, p->k, x, norm_weight, p->eps,
               nullptr, nullptr};
    // (a non-null table selects the epilogue; with rotate = 0 it is not read)
    g.table = rope_table ? rope_table : x;
    g.state = state;
    g.k_cache = k_cache;
    g.v_cache = v_cache;
    g.row0 = p->row0;
    g.q_rows = static_cast<uint32_t>(q_rows);
    g.kv_rows = static_cast<uint32_t>(kv_rows);
    g.hd = p->head_dim;
    g.capacity = p->capacity;
    g.kv_f16 = p->kv_type == VKML_F16;
    g.rotate = p->rotate;
    return dispatch_format<kStore, 1>(p->b_type, p->scale_type, g, "gemv_rope");
}

int vkml_gemv(const vkml_gemv_params* p, const float* a, const void* b, float* out, const void* b_scales) {
    VKML_REQUIRE_INIT();
    VKML_CHECK_ARG(p, "gemv: null params");
    VKML_CHECK_ARG(p->m >= 1 && p->m <= 8, "gemv: m must be 1 to 8, got " + std::to_string(p->m));
    VKML_CHECK_ARG(p->b_type <= VKML_Q4_K, "gemv: unknown weight type " + std::to_string(p->b_type));
    const uint32_t batches = std::max(p->batches, 1u), group = std::max(p->b_group, 1u);
    VKML_CHECK_ARG(batches <= 65535, "gemv: too many batches");
    if (p->b_type >= VKML_Q8_0) {
        const uint32_t unit = p->b_type == VKML_Q4_K ? 256 : 32;
        VKML_CHECK_ARG(p->k % unit == 0, "gemv: k = " + std::to_string(p->k) + " is not whole blocks of " + std::to_string(unit));
        VKML_CHECK_ARG(b_scales, "gemv: quantized weights need scales");
        VKML_CHECK_ARG(batches == 1, "gemv: batches need a float b");
    }
    if (p->n == 0) return VKML_OK;
    VKML_CHECK_ARG(a && b && out, "gemv: null buffer");
    const dim3 grid((p->n + 7) / 8, batches);
    vkml::abi::ProfileScope prof("gemv");
    // Whole, aligned groups of four in a's rows and a float b's.
    const uint32_t unit = p->b_type == VKML_F32 ? 16 : 8;
    if (p->b_type <= VKML_BF16 && p->k % 4 == 0 && p->k > 0 && p->b_stride % 4 == 0 && reinterpret_cast<uintptr_t>(a) % 16 == 0 &&
        reinterpret_cast<uintptr_t>(b) % unit == 0) {
        if (p->b_type == VKML_F32) launch_float4<VKML_F32>(*p, a, b, out, batches, group);
        else if (p->b_type == VKML_F16) launch_float4<VKML_F16>(*p, a, b, out, batches, group);
        else launch_float4<VKML_BF16>(*p, a, b, out, batches, group);
        return vkml::abi::check_launch("gemv");
    }
    hipStream_t s = vkml::abi::stream();
    const uint64_t bst = p->b_stride;
#define VKML_GEMV_LAUNCH(T) \
    hipLaunchKernelGGL(k_gemv_float<T>, grid, dim3(256), 0, s, a, p->m, b, b_scales, p->scale_type, out, p->n, p->k, group, bst)
    switch (p->b_type) {
        case VKML_F32: VKML_GEMV_LAUNCH(VKML_F32); break;
        case VKML_F16: VKML_GEMV_LAUNCH(VKML_F16); break;
        case VKML_BF16: VKML_GEMV_LAUNCH(VKML_BF16); break;
        case VKML_Q8_0: VKML_GEMV_LAUNCH(VKML_Q8_0); break;
        case VKML_Q4_0: VKML_GEMV_LAUNCH(VKML_Q4_0); break;
        case VKML_Q4_1: VKML_GEMV_LAUNCH(VKML_Q4_1); break;
        default: VKML_GEMV_LAUNCH(VKML_Q4_K); break;
    }
#undef VKML_GEMV_LAUNCH
    return vkml::abi::check_launch("gemv");
}

}  // extern "C"
