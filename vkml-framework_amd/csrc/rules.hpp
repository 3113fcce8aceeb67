// rules.hpp -- which kernel of a family a call takes, where that follows from
// its sizes and addresses alone: host code without HIP, so that the choices
// can be checked on any machine. What each line rests on stands beside it.
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

}  // namespace vkml::rules
