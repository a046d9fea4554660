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
    float alpha, beta;
    // the feature steps are divided over k_splits workgroups per output tile, which store f32 partial tiles
    // [split][m][n_total]; gemm_finish_kernel adds them up in split order and applies the write stage
    uint32_t k_splits, steps_per_split, n_total;
    float *partial;
    RopeDev rope;
    uint32_t page_shift;  // log2 of rope.block_size, 32 = not a power of two
};

// Rotation of the piece hd .. hd + 7 of a head: the first table column that it takes, the columns (adjacent pairs (hd + 2i, hd + 2i + 1):
// 4 of them, from hd / 2; pairs (hd, hd + D / 2): 8, from hd mod D / 2), and the piece rotated with them.
__device__ __forceinline__ uint32_t rope_column(const RopeDev &r, uint32_t hd) { return r.normal ? hd >> 1 : hd & ((r.head_dim >> 1) - 1u); }
__device__ __forceinline__ void rope_columns(const RopeDev &r, uint32_t table_row, uint32_t column, h8_t &c, h8_t &s) {
    typedef _Float16 h4v_t __attribute__((ext_vector_type(4)));
    const size_t at = (size_t)table_row * (r.head_dim >> 1) + column;
    if (r.normal) {
        const h4v_t c4 = fa_norm::load_global<h4v_t>(r.cos_t + at), s4 = fa_norm::load_global<h4v_t>(r.sin_t + at);
        c = __builtin_shufflevector(c4, c4, 0, 1, 2, 3, 0, 1, 2, 3), s = __builtin_shufflevector(s4, s4, 0, 1, 2, 3, 0, 1, 2, 3);
    } else {
        c = fa_norm::load_global<h8_t>(r.cos_t + at), s = fa_norm::load_global<h8_t>(r.sin_t + at);
    }
}
__device__ __forceinline__ h8_t rope_piece(const RopeDev &r, h8_t y, h8_t mate, h8_t c, h8_t s, bool first) {
    h8_t o;
    if (r.normal) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[2 * i] = (_Float16)rope_one((float)y[2 * i], (float)y[2 * i + 1], (float)c[i], (float)s[i], true);
            o[2 * i + 1] = (_Float16)rope_one((float)y[2 * i + 1], (float)y[2 * i], (float)c[i], (float)s[i], false);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (_Float16)rope_one((float)y[e], (float)mate[e], (float)c[e], (float)s[e], first);
    }
    return o;
}

// Write stage of one piece: y = the projections of token gm, columns gn .. gn + 7 of matrix mat (0 Q, 1 K, 2 V),
// already rounded to f16 as FusedQkv stores them; mate = the piece half a head away (NeoX pairing; unused otherwise).
// Q goes to q_rot[h][gm][hd], K (rotated) and V (as is) to cache row position_offset + gm of KV head h.
__device__ __forceinline__ void rope_store_piece(const GemmDev &a, int mat, uint32_t gm, uint32_t gn, h8_t y, const h8_t mate) {
    const RopeDev &r = a.rope;
    const uint32_t D = r.head_dim, half = D >> 1, h = gn / D, hd = gn - h * D;
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
        h8_t c, s;
        rope_columns(r, tp, rope_column(r, hd), c, s);
        y = rope_piece(r, y, mate, c, s, hd < half);
    }
    *reinterpret_cast<h8_t *>(dst) = y;
}

typedef unsigned int u4v_t __attribute__((ext_vector_type(4)));
typedef _Float16 h2v_t __attribute__((ext_vector_type(2)));

}  // namespace fa_gemm
