// RMSNorm pieces shared by the projection kernels (src/metals/rmsnorm/rmsnorm.metal:17-96, qkv_project.metal:48-67), and the
// lane sums they and the weight streams use.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace fa_norm {

typedef _Float16 norm_h8_t __attribute__((ext_vector_type(8)));
typedef uint32_t norm_u4_t __attribute__((ext_vector_type(4)));
typedef unsigned int norm_u2_t __attribute__((ext_vector_type(2)));

// A load from device memory through an address that is chosen per lane. (The compiler does not see that such a pointer - a select
// between arguments - is to global memory and would use flat loads, which also count as LDS accesses: every wait for one is a
// wait for both.)
template <typename T>
__device__ __forceinline__ T load_global(const void *p) {
    return *(const __attribute__((address_space(1))) T *)(uintptr_t)p;
}
template <typename T>
__device__ __forceinline__ T load_global_once(const void *p) {  // read once per launch: not kept in the caches
    return __builtin_nontemporal_load((const __attribute__((address_space(1))) T *)(uintptr_t)p);
}

template <typename T>
__device__ __forceinline__ void store_global(void *p, T v) {
    *(__attribute__((address_space(1))) T *)(uintptr_t)p = v;
}

// 1 / sqrt(mean + eps) from a row's sum of squares: one hardware reciprocal square root (within an ulp; the library's rsqrtf
// adds a rescaling of denormal arguments, which epsilon keeps away from here; of a million normalised f16 values 50 to 65 are not
// the rounding of the exact quotient, 75 to 100 with a division and the library's function). The empty slots: an instruction that uses a
// transcendental's result must not follow at once; the compiler sees to that by itself, but not in front of scale8's assembly.
__device__ __forceinline__ float inv_rms(float sum_sq, float inv_k, float eps) {
    float r = __builtin_amdgcn_rsqf(fmaf(sum_sq, inv_k, eps));
    asm volatile("s_nop 1" : "+v"(r));
    return r;
}

// v + the values of lanes l ^ 16, l ^ 32, l ^ 48, in every lane
__device__ __forceinline__ float sum_rows_of_16(float v) {
    norm_u2_t t = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(t.x) + __uint_as_float(t.y);
    t = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(t.x) + __uint_as_float(t.y);
}

// Sum over the wave's 64 lanes in every lane: rotations within 16 lanes, then swaps of lane groups - vector instructions all
// the way (through __shfl_xor each of the six steps is a trip through the LDS crossbar, one after the other).
__device__ __forceinline__ float wave_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, true));  // row_ror:8
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xf, 0xf, true));  // row_ror:4
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x122, 0xf, 0xf, true));  // row_ror:2
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x121, 0xf, 0xf, true));  // row_ror:1
    return sum_rows_of_16(v);
}

// (x * inv_rms) * gamma, each product rounded to f32, the result to f16: two instructions per element that take the f16 halves
// as they lie in the registers (the plain form converts both factors and the result separately, five per element).
__device__ __forceinline__ norm_h8_t scale8(norm_h8_t x, float inv_rms, norm_h8_t gamma) {
    const norm_u4_t x2 = __builtin_bit_cast(norm_u4_t, x), g2 = __builtin_bit_cast(norm_u4_t, gamma);
    const float neg_zero = -0.0f;  // (a sum with -0 keeps the sign of a zero product)
    norm_u4_t y2;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float t0, t1;
        uint32_t y;
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(t0) : "v"(x2[e]), "v"(inv_rms), "v"(neg_zero));
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(t1) : "v"(x2[e]), "v"(inv_rms), "v"(neg_zero));
        asm("v_fma_mixlo_f16 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[0,1,0]" : "=v"(y) : "v"(t0), "v"(g2[e]), "v"(neg_zero));
        asm("v_fma_mixhi_f16 %0, %1, %2, %3 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "+v"(y) : "v"(t1), "v"(g2[e]), "v"(neg_zero));
        y2[e] = y;
    }
    return __builtin_bit_cast(norm_h8_t, y2);
}

}  // namespace fa_norm
