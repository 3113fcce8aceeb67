// The dispatch rules of csrc/rules.hpp as C functions, for test_rules.py.
#include "rules.hpp"

using namespace vkml::rules;

extern "C" int float_loads_c(const vkml_matmul_params* p, uint64_t a, uint64_t b) { return float_loads(*p, a, b); }

// 10 r + nc
extern "C" int wave_tile_c(const vkml_matmul_params* p) { return 10 * wave_tile(*p).r + wave_tile(*p).nc; }

extern "C" int cut_last_chunk_c(const vkml_matmul_params* p) { return cut_last_chunk(*p); }

extern "C" uint32_t rows_chunk_c(uint32_t k) { return rows_chunk(k); }

extern "C" int gemv_row_each_c(uint32_t m, uint32_t n, uint32_t batches) { return gemv_row_each(m, n, batches); }

extern "C" int gemv_row_cached_c(const vkml_gemv_params* p) { return gemv_row_cached(*p); }

extern "C" int dot_tail_c(int rt, int ct, uint32_t k) { return dot_tail(rt, ct, k); }

// 10 rt + ct
extern "C" int dot_tile_c(uint32_t b_type, int f16_scales, uint32_t m, uint32_t n) {
    const DotTile t = dot_tile(b_type, f16_scales != 0, m, n);
    return 10 * t.rt + t.ct;
}

extern "C" int wide_blocks_c(const vkml_attend_prompt_params* p, uint32_t workgroups, uint32_t compute_units) {
    return wide_blocks(*p, workgroups, compute_units);
}

// The tiles of a launch in the order of its workgroups, 65536 row + col, ~0 for none; the number of workgroups.
extern "C" uint32_t dot_bands_c(uint32_t rows, uint32_t columns, uint32_t* tiles) {
    const DotBands b = dot_bands(rows, columns);
    if (b.width == 0) return 0;
    for (uint32_t i = 0; i < 8 * b.share; ++i) {
        uint32_t row, col;
        tiles[i] = b.tile(i, row, col) ? 65536 * row + col : ~0u;
    }
    return 8 * b.share;
}
