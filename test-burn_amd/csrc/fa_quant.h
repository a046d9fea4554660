// Block-quantised weights as f16, exactly and without a conversion per element: a byte u behind 0x64 is the f16 1024 + u, so four
// weights take two byte permutes and one packed subtraction.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace fa_quant {

typedef _Float16 quant_h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 quant_h8_t __attribute__((ext_vector_type(8)));

// Eight bytes, each u with the bits of `flip` turned over -> 1024 + u - off
__device__ __forceinline__ quant_h8_t bytes_to_f16(uint32_t a, uint32_t b, uint32_t flip, _Float16 off) {
    const quant_h2_t bias = {off, off};
    quant_h8_t r;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t u = (i ? b : a) ^ flip;
        const quant_h2_t lo = __builtin_bit_cast(quant_h2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x05010400u)) - bias;
        const quant_h2_t hi = __builtin_bit_cast(quant_h2_t, __builtin_amdgcn_perm(0x64646464u, u, 0x07030602u)) - bias;
        r[4 * i] = lo[0], r[4 * i + 1] = lo[1], r[4 * i + 2] = hi[0], r[4 * i + 3] = hi[1];
    }
    return r;
}

// Eight Q8_0 weights: s + 128 is a byte. AHEAD: both words turned over ahead of the permutes, as the weight streams have it; the tile
// kernels lose 1 % with that order (500 rows, 1152 x 896: 9.24 -> 9.31 us).
template <bool AHEAD = false>
__device__ __forceinline__ quant_h8_t q8_to_f16(uint32_t a, uint32_t b) {
    constexpr uint32_t FLIP = 0x80808080u;
    return AHEAD ? bytes_to_f16(a ^ FLIP, b ^ FLIP, 0u, (_Float16)1152.0f) : bytes_to_f16(a, b, FLIP, (_Float16)1152.0f);
}

// Eight Q4_0 weights (element 2i in the low nibble of byte i, value = nibble - 8: policy_q4_0.metal:70-86): the nibbles become two
// words of four bytes in element order.
__device__ __forceinline__ quant_h8_t q4_to_f16(uint32_t w) {
    const uint32_t even = w & 0x0f0f0f0fu, odd = (w >> 4) & 0x0f0f0f0fu;
    return bytes_to_f16(__builtin_amdgcn_perm(odd, even, 0x05010400u), __builtin_amdgcn_perm(odd, even, 0x07030602u), 0u, (_Float16)1032.0f);
}

}  // namespace fa_quant
