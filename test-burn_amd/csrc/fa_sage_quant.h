// The int8 quantiser of the smoothed K rows: q = clamp(rint(x / scale), -127, 127), 0 when the scale is not positive
// (docs/SAGE.md:51-65 leaves the rounding open; the CPU oracle's is this one), and -127 where the quotient is no number. A 32-row
// block shares one scale, an f16 value, so a block's thousands of quotients have one divisor, and the division is what the
// quantising kernels spend their time on. SageDivisor does the divisor's share once: the reciprocal estimate and its refinement,
// exactly as the compiler's own expansion of an f32 division computes them. Per quotient that leaves q0 = x r and the step
// q = q0 + (x - d q0) r with fused multiply-adds, which end at the correctly rounded quotient: the same value `x / scale` gives, bit
// for bit. One such step is enough here, where the expansion takes two, because the divisor is an f16 value, 11 bits: the
// refined reciprocal is then the correctly rounded one (1 - d r0 is exact, and 1 / d is too far from the middle of two floats for what
// is left of the error), x - d q0 is exact, and x / d is 2^-12 units in the last place or more away from the middle of two floats
// (on it, it would have more bits than x has), where the step's error is 2^-23. The expansion's rescaling of extreme operands does
// not come into play for a divisor that is a finite f16 value, 2^-24 .. 65504, and numerators of a block whose largest
// magnitude made that divisor: tests/test_sage_division.py checks the sequence on the CPU against the division for every such
// divisor, with the estimate off by an ulp either way, on quotients next to the rounding boundaries of the quantiser. The same for a
// query's scale, an f32 value that is an f16 value / 127, and the f16 values up to it.
// Scales that are no such divisor need no other path: with d = r = 0 a number's quotient is 0 and that of an infinity or a NaN is no
// number, which is what an infinite scale gives; and with clamps of 0 as well it is 0 for all, as for a scale that is not positive.
#pragma once
#include <hip/hip_runtime.h>

struct SageDivisor {
    float d, r, bound;
};

__device__ __forceinline__ SageDivisor sage_divisor(float d) {
    const float r0 = __builtin_amdgcn_rcpf(d);
    const float e = __builtin_fmaf(-d, r0, 1.0f);
    const bool finite = d > 0.0f && d < __builtin_inff();
    return SageDivisor{finite ? d : 0.0f, finite ? __builtin_fmaf(e, r0, r0) : 0.0f, d > 0.0f ? 127.0f : 0.0f};
}

// The int8 value in the low byte: the quotient clamped (a NaN gives the lower bound) and rounded to an integer, half to even, by
// adding 1.5 * 2^23, whose sum holds the integer in its low bits in two's complement.
__device__ __forceinline__ uint32_t sage_quant_byte(float x, const SageDivisor &v) {
    const float q0 = x * v.r;
    const float q = __builtin_fmaf(__builtin_fmaf(-v.d, q0, x), v.r, q0);
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_fmed3f(q, -v.bound, v.bound) + 12582912.0f);
}

// Four values -> four int8 in a word (value i in byte i). Six instructions per value with its share of the packing; with a
// second step, a rounding, two for the clamp and a conversion they were nearly ten. (A decode step of SmolLM3 at 300 / 8000 / 20000 /
// 32768 keys, the query and the difference from the mean likewise: 10.1 -> 8.4, 11.3 -> 9.8, 11.5 -> 10.2, 13.9 -> 13.6 us.)
__device__ __forceinline__ uint32_t sage_quant4_i8(float x0, float x1, float x2, float x3, const SageDivisor &v) {
    const uint32_t lo = __builtin_amdgcn_perm(sage_quant_byte(x1, v), sage_quant_byte(x0, v), 0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm(sage_quant_byte(x3, v), sage_quant_byte(x2, v), 0x0c0c0400u);
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// max(m, |a|, |b|), NaNs passed over; and k - mu for the two f16 values of a word: the difference of a widened f16 value and an f32
// one, one rounding. One instruction each, which the compiler makes two or three of.
__device__ __forceinline__ float sage_max3(float m, float a, float b) {
    float r;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float sage_lo_minus(uint32_t word, float mu) {
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(word), "v"(mu));
    return r;
}
__device__ __forceinline__ float sage_hi_minus(uint32_t word, float mu) {
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(word), "v"(mu));
    return r;
}
