// What the GEMM kernels of FusedQkv / MatMul share (fa_gemm.hip, fa_tile_*.hip): the launch's description, the RoPE write stage, the
// conversion of block-quantised weights, and how the tile kernels are launched.
#pragma once
#include "fa_internal.h"
#include "fa_norm.h"
#include "fa_qkv_rope.h"
#include "fa_quant.h"

namespace fa_gemm {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4v_t __attribute__((ext_vector_type(4)));
typedef float f16v_t __attribute__((ext_vector_type(16)));

struct GemmDev {
    const void *w[3];       // f16, or int8 (Q8_0) / nibbles (Q4_0) in the same element order
    const __half *scales[3];  // Q8_0: f16 [rows, k_dim / 32] per matrix
    const __half *bias[3];
    __half *out[3];
    uint32_t rows[3];       // weight rows per matrix
    uint32_t tiles[3];      // tiles per matrix, of the width that the launch takes
    const __half *x;        // [m, k_dim] (already normalised when the op has a gamma)
    const __half *residual; // nullable, [m, rows[0]]
    uint32_t k_dim, m, m_tiles, n_tiles, canonical, vec_store;
    uint32_t panel_inv;     // fa_inverse(input tiles x weight tiles that are gone through together)
    float alpha, beta;
    // the feature steps are divided over k_splits workgroups per output tile, which store f32 partial tiles
    // [split][m][n_total]; gemm_finish_kernel adds them up in split order and applies the write stage
    uint32_t k_splits, steps_per_split, n_total;
    float *partial;
    RopeDev rope;
    uint32_t page_shift;  // log2 of rope.block_size, 32 = not a power of two
};

typedef _Float16 h4v_t __attribute__((ext_vector_type(4)));

// x * c - mate * s (`first`), or x * c + mate * s, of f16 values: the products are exact in f32, so one rounded sum of an exact product and
// another is what rope_one gives, in two instructions that take the f16 halves as they lie in the registers.
template <int X, int M, int C>
__device__ __forceinline__ float rope_mix(uint32_t x, uint32_t mate, uint32_t c, uint32_t s, bool first) {
    const float neg_zero = -0.0f;  // (a sum with -0 keeps the sign of a zero product)
    float t;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[%4,%5,0] op_sel_hi:[1,1,0]" : "=v"(t) : "v"(mate), "v"(s), "v"(neg_zero), "n"(M), "n"(C));
    if (first) asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[%4,%5,0] op_sel_hi:[1,1,0]" : "=v"(t) : "v"(x), "v"(c), "v"(t), "n"(X), "n"(C));
    else asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[%4,%5,0] op_sel_hi:[1,1,0]" : "=v"(t) : "v"(x), "v"(c), "v"(t), "n"(X), "n"(C));
    return t;
}
typedef uint32_t rope_u4_t __attribute__((ext_vector_type(4)));
typedef uint32_t rope_u2_t __attribute__((ext_vector_type(2)));
// Rotation of a piece of 8 dims whose pairs are (2i, 2i + 1): 4 table columns
__device__ __forceinline__ h8_t rope_adjacent(h8_t y, h4v_t c4, h4v_t s4) {
    const rope_u4_t y2 = __builtin_bit_cast(rope_u4_t, y);
    const rope_u2_t c = __builtin_bit_cast(rope_u2_t, c4), s = __builtin_bit_cast(rope_u2_t, s4);
    h8_t o;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        o[4 * i] = (_Float16)rope_mix<0, 1, 0>(y2[2 * i], y2[2 * i], c[i], s[i], true), o[4 * i + 1] = (_Float16)rope_mix<1, 0, 0>(y2[2 * i], y2[2 * i], c[i], s[i], false);
        o[4 * i + 2] = (_Float16)rope_mix<0, 1, 1>(y2[2 * i + 1], y2[2 * i + 1], c[i], s[i], true), o[4 * i + 3] = (_Float16)rope_mix<1, 0, 1>(y2[2 * i + 1], y2[2 * i + 1], c[i], s[i], false);
    }
    return o;
}
// ... whose pairs are half a head apart, `mate` the piece there: 8 columns; `first`: the piece is of the first half
__device__ __forceinline__ h8_t rope_apart(h8_t y, h8_t mate, h8_t c8, h8_t s8, bool first) {
    const rope_u4_t x = __builtin_bit_cast(rope_u4_t, y), m = __builtin_bit_cast(rope_u4_t, mate), c = __builtin_bit_cast(rope_u4_t, c8);
    rope_u4_t s = __builtin_bit_cast(rope_u4_t, s8);
    h8_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t sgn = first ? s[i] ^ 0x80008000u : s[i];
        o[2 * i] = (_Float16)rope_mix<0, 0, 0>(x[i], m[i], c[i], sgn, false), o[2 * i + 1] = (_Float16)rope_mix<1, 1, 1>(x[i], m[i], c[i], sgn, false);
    }
    return o;
}
// Rotation of the piece hd .. hd + 7 of a head from the tables' row
__device__ __forceinline__ h8_t rope_piece(const RopeDev &r, uint32_t table_row, uint32_t hd, h8_t y, h8_t mate) {
    const uint32_t half = r.head_dim >> 1, column = r.normal ? hd >> 1 : hd & (half - 1u);
    const size_t at = (size_t)table_row * half + column;
    if (r.normal) return rope_adjacent(y, fa_norm::load_global<h4v_t>(r.cos_t + at), fa_norm::load_global<h4v_t>(r.sin_t + at));
    return rope_apart(y, mate, fa_norm::load_global<h8_t>(r.cos_t + at), fa_norm::load_global<h8_t>(r.sin_t + at), hd < half);
}

// Write stage of one piece: y = the projections of token gm, columns gn .. gn + 7 of matrix mat (0 Q, 1 K, 2 V),
// already rounded to f16 as FusedQkv stores them; mate = the piece half a head away (NeoX pairing; unused otherwise).
// Q goes to q_rot[h][gm][hd], K (rotated) and V (as is) to cache row position_offset + gm of KV head h.
__device__ __forceinline__ void rope_store_piece(const GemmDev &a, int mat, uint32_t gm, uint32_t gn, h8_t y, const h8_t mate) {
    const RopeDev &r = a.rope;
    const uint32_t D = r.head_dim, h = gn / D, hd = gn - h * D;
    const uint32_t pos = r.position_offset + gm;
    __half *dst;
    if (mat == 0) {
        dst = a.out[0] + ((size_t)h * a.m + gm) * D + hd;
    } else {
        if (pos >= r.capacity) return;  // never outside the cache
        size_t row;
        if (!r.block_table) {
            row = ((size_t)h * r.max_seq_len + pos) * D;
        } else {
            const size_t blk = (size_t)r.block_table[pos / r.block_size];
            row = ((blk * r.n_kv_heads + h) * r.block_size + pos % r.block_size) * D;
        }
        dst = (mat == 1 ? a.out[1] : a.out[2]) + row + hd;
    }
    if (mat != 2 && r.apply) {
        const uint32_t tp = pos < r.table_rows ? pos : r.table_rows - 1;  // stay inside the tables
        y = rope_piece(r, tp, hd, y, mate);
    }
    *reinterpret_cast<h8_t *>(dst) = y;
}

typedef unsigned int u4v_t __attribute__((ext_vector_type(4)));
typedef _Float16 h2v_t __attribute__((ext_vector_type(2)));

}  // namespace fa_gemm
