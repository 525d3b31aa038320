// polar_norm.hpp — the normalisation's arithmetic and summation order, shared by the
// element-wise passes (polar_norm.hip) and the resident kernel (polar_resident.hip).
#pragma once

#include "polar_tile.hpp"

namespace muon_polar {

__device__ __forceinline__ float bf16_round(float v) {
    return bf16_bits_to_f32(f32_to_bf16_bits(v));
}

// Sum of v over a wave, the same in every lane (butterfly in a fixed order).
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// The recipe's divisor bf16(bf16(norm · 1.01) + 1e-6) from the sum of squares.
__device__ __forceinline__ float norm_divisor(float total) {
    const float norm = bf16_round(sqrtf(total));
    return bf16_round(bf16_round(norm * 1.01f) + 1e-6f);
}

// Two bf16 values in one word: squares added to acc, low half first.
__device__ __forceinline__ float add_squares(float acc, uint32_t w) {
    const float lo = bf16_bits_to_f32(w & 0xffffu), hi = bf16_bits_to_f32(w >> 16);
    return fmaf(hi, hi, fmaf(lo, lo, acc));
}

}  // namespace muon_polar
