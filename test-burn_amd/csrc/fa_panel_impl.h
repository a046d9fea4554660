// The panel kernel (see fa_panel.h) and its launcher for one weight width.
#pragma once
#include <atomic>

#include "fa_panel.h"
#include "fa_quant.h"

namespace fa_panel {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef float f4v_t __attribute__((ext_vector_type(4)));
typedef unsigned int u2v_t __attribute__((ext_vector_type(2)));
typedef unsigned int u4v_t __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ T pick3(int mat, T x0, T x1, T x2) {
    return mat == 0 ? x0 : mat == 1 ? x1 : x2;
}

__device__ __forceinline__ float dot8_self(h8_t a, float acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_fdot2(h2_t{a[2 * i], a[2 * i + 1]}, h2_t{a[2 * i], a[2 * i + 1]}, acc, false);
    return acc;
}

// Weight width -> what a lane holds of 8 consecutive weights, and those as f16 (times the block's scale, rounded to f16).
template <int WB>
struct Weights;
template <>
struct Weights<16> {
    typedef h8_t raw_t;
    static __device__ __forceinline__ h8_t f16(raw_t w, _Float16) { return w; }
    static __device__ __forceinline__ h8_t plain(raw_t w) { return w; }
    static __device__ __forceinline__ raw_t part(raw_t w, int) { return w; }
};
template <>
struct Weights<8> {
    typedef u2v_t raw_t;
    static __device__ __forceinline__ raw_t part(u4v_t w, int i) { return raw_t{w[2 * i], w[2 * i + 1]}; }  // 8 weights of 16
    static __device__ __forceinline__ h8_t plain(raw_t w) { return fa_quant::q8_to_f16<true>(w[0], w[1]); }
    static __device__ __forceinline__ h8_t f16(raw_t w, _Float16 s) { return plain(w) * h8_t{s, s, s, s, s, s, s, s}; }
};
template <>
struct Weights<4> {
    typedef uint32_t raw_t;
    static __device__ __forceinline__ raw_t part(u4v_t w, int i) { return w[i]; }  // 8 weights of 32
    static __device__ __forceinline__ h8_t plain(raw_t w) { return fa_quant::q4_to_f16(w); }
    static __device__ __forceinline__ h8_t f16(raw_t w, _Float16 s) { return plain(w) * h8_t{s, s, s, s, s, s, s, s}; }
};

// What a lane reads in the place of an F16 weight block past the row's last.
static __device__ const h8_t zero_weights = {0, 0, 0, 0, 0, 0, 0, 0};

// FEW: at most 8 input rows to a workgroup, one per wave - the launch has no more, or (EIGHTS) they are one of its passes: the other half of
// the 16 columns is not loaded, normalised or stored. (8 rows, two per wave -> one: QKV with its norm, 5120 x 3072 F16 10.1 -> 9.3 us, Q8_0
// 10.1 -> 9.0, Q4_0 10.0 -> 8.3; 1152 x 896 F16 4.8 -> 4.4; 3072 x 3072 without a norm 6.5 -> 5.8, 6.0 -> 5.5, 6.4 -> 5.1.)
template <int WB, int NT, int NC, int PK, bool ROPE, bool SUMS, bool FEW, bool EIGHTS, bool WALK>
__global__ void __launch_bounds__(NTHREADS, (two_per_cu(NT, NC, PK, ROPE) ? 4 : 2)) panel_kernel(PanelDev a_by_value) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    static_assert(std::is_trivially_copyable<PanelDev>::value, "read as raw bytes from the argument block, where it is the first member");
    const PanelDev &a = *(const PanelDev *)__builtin_amdgcn_kernarg_segment_ptr();
    (void)a_by_value;
    typedef Weights<WB> W;
    typedef typename W::raw_t raw_t;
    constexpr int XROW = row_bytes<PK>(), NR = FEW ? 1 : 2 * NC, NB = 2 * PK;
    static_assert(!FEW || NC == 1, "one group of input rows");
    constexpr uint32_t PASS = FEW ? 8 : NC * 16;  // input rows of a pass
    constexpr bool WIDE = WB != 16 && !SUMS, TURN = TURNS<WB, PK, SUMS>;
    constexpr int GB = !WIDE && !TURN ? 1 : WB == 8 ? 2 : 4, NQ = NB / GB;  // blocks per request, requests per tile
    typedef typename std::conditional<WIDE || TURN, u4v_t, raw_t>::type req_t;
    // A wave that asks for more than the memory takes stands still until it has (a workgroup of 32 rows of 3072 features asks for
    // 3 us), and normalises no rows meanwhile. RING, of the longest rows, whose workgroups have one pass each: it asks for the first NF
    // requests of a tile, and for another whenever one has been multiplied - REST: for all others when the rows are in LDS (F16, 9 rows
    // of 3072 features: 4.9 us, one by one 5.1). All tiles' first requests come before any second one. FusedQkv of 5120 x 3072, all asked
    // for at once tile after tile -> this, us: F16 2 rows 9.7 -> 8.4, 16 rows 10.8 -> 9.7; Q8_0 9.1 -> 7.7, 11 rows 10.6 -> 9.2; Q4_0,
    // whose requests are few and all made at once, 8.7 -> 8.2.
    // WALK, of the longest rows: workgroups that go on to further passes keep all their weights. SPLIT: some of them, too, ask for a
    // tile's other requests when the first pass's rows are in LDS (o_proj of 3072 x 3072 Q8_0 24 and 32 rows 7.1 -> 6.2 us).
    static_assert(!WALK || PK > 4, "shorter rows have one kernel for both");
    constexpr bool RING = PK > 4 && !WALK, SPLIT = WALK && (WB == 8 ? !ROPE || NT == 2 : WB == 16 && !ROPE && NT == 1);
    constexpr bool REST = (RING && WB == 16 && NT == 1) || SPLIT;
    constexpr int NF = SPLIT ? (NT == 1 ? (NQ < 8 ? NQ : 8) : 4)
                       : !RING || WB == 4 ? NQ : WB == 16 ? (NT <= 2 ? 8 : NT == 3 ? 6 : 4) : NT == 1 ? (NQ < 8 ? NQ : 8) : NT == 2 ? 4 : NT == 3 ? 3 : 2;
    constexpr int NA = REST ? NQ : NF;  // places in registers
    // The order of the first requests is input rows, the norm's weights, scales, weights. Loads complete in the order in which they
    // are issued; left to itself the compiler puts the weights ahead of the rows in most of the kernels, and what is done with
    // the rows then waits for the whole weight stream. (m 12 .. 32, K 2048 .. 3072: o_proj 4 to 14 % less. With the longest rows and a
    // norm of two rows per wave the norm's chain is longer than the weights' stream, and the compiler's mixture is 1 to 3 % better.)
    constexpr bool ORDERED = FEW || !ROPE || PK <= 4 || (WALK ? SPLIT : WB == 8 || NT > 2);
    const unsigned char *const w0 = a.w[0], *const w1 = a.w[1], *const w2 = a.w[2];
    const uint32_t rows0 = a.rows0, rows1 = a.rows1, total_rows = a.total_rows;
    const __half *const x_in = a.x, *const gamma = a.gamma;
    constexpr bool BESIDE = NC == 1 && (!FEW || EIGHTS) && !WALK;  // (the branch in the others takes 3 to 5 % of a short launch)
    const uint32_t beside = BESIDE || RING ? a.beside : 0, inv_beside = BESIDE || RING ? a.inv_beside : 0;
    const uint32_t K = a.k_dim, m_rows = a.m, rows_per_wg = a.rows_per_wg, canonical_u = a.canonical, n_pass = a.n_pass;
    const __half *const sp0 = a.scales[0], *const sp1 = a.scales[1], *const sp2 = a.scales[2];
    const uint32_t normal = a.r.normal, head_dim = a.r.head_dim, scale_pairs = a.scale_pairs;
    // (the launch's arguments in two trips through the scalar cache: what the first requests need, and the rest behind them)
    asm volatile("" ::"s"(w0), "s"(w1), "s"(w2), "s"(rows0), "s"(rows1), "s"(total_rows), "s"(x_in), "s"(gamma), "s"(K), "s"(m_rows),
                 "s"(rows_per_wg), "s"(canonical_u), "s"(n_pass));
    if constexpr (BESIDE || RING) asm volatile("" ::"s"(beside), "s"(inv_beside));
    if constexpr (WB != 16) asm volatile("" ::"s"(sp0), "s"(sp1), "s"(sp2), "s"(scale_pairs));
    if constexpr (ROPE) asm volatile("" ::"s"(normal), "s"(head_dim));
    const bool canonical = canonical_u != 0;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, c = lane >> 4;
    const uint32_t nkb = K / 32, n_pieces = K / 8;
    uint32_t along = blockIdx.x, first_pass = blockIdx.y, pass_step = gridDim.y;
    if (RING || (BESIDE && beside)) {
        const uint32_t eighth = blockIdx.x >> 3, group = fa_quotient(eighth, beside, inv_beside);
        along = group * 8 + (blockIdx.x & 7), first_pass = eighth - group * beside, pass_step = beside;
    }
    const uint32_t row_begin = along * rows_per_wg;
    const uint32_t row_end = min(total_rows, row_begin + rows_per_wg);
    if (row_begin >= row_end) return;
    // ROPE (rows_per_wg is even, the matrices hold whole heads): the pairing and the head size
    uint32_t neox = 0, half_shift = 0, pair_begin = 0, pair_end = 0;
    if constexpr (ROPE) {
        neox = normal ? 0u : 1u, half_shift = head_dim == 128 ? 6u : 5u;
        pair_begin = row_begin >> 1, pair_end = row_end >> 1;
    }
    // Weight row of slot (tile t, row n of the tile) across the three matrices laid end to end; a slot past the workgroup's
    // last row gives the workgroup's first row with valid = false. NeoX pairs: tiles 0 and 2 (of an odd number the last tile's first 8
    // rows) hold rows of first halves of heads, tiles 1 and 3 (the other 8) their mates half a head on.
    auto slot_row = [&](uint32_t t, uint32_t n_, bool &valid) __attribute__((always_inline)) -> uint32_t {
        if (ROPE && neox) {
            const bool both = NT % 2 == 1 && t == NT - 1;
            const uint32_t p = pair_begin + 16u * (t >> 1) + (both ? n_ & 7u : n_), pv = p < pair_end ? p : pair_begin;
            valid = p < pair_end;
            return ((pv >> half_shift) << (half_shift + 1)) + (pv & ((1u << half_shift) - 1u)) + ((both ? n_ >> 3 : t & 1u) << half_shift);
        }
        const uint32_t gr = row_begin + 16u * t + n_;
        valid = gr < row_end;
        return valid ? gr : row_begin;
    };
    auto locate = [&](uint32_t row, int &mat) __attribute__((always_inline)) -> uint32_t {
        const bool in1 = row >= rows0, in2 = row >= rows0 + rows1;
        mat = (in1 ? 1 : 0) + (in2 ? 1 : 0);
        return row - (in2 ? rows0 + rows1 : in1 ? rows0 : 0u);
    };

    // ---- input rows of a pass: rows wave, wave + 8, ... of it (a row past the chunk's last re-reads the last: its column is not
    // stored), piece j of a row = features 512 j + 8 lane ..
    h8_t xr[NR][PK];
    auto request_rows = [&](uint32_t pass, bool first) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            if (i > (first ? 1 : 0) && pass * PASS + 8u * i >= m_rows) break;  // (uniform: no such rows in the pass; the first one is not waited for)
            const __half *row = x_in + (size_t)min(pass * PASS + (uint32_t)wave + 8u * i, m_rows - 1u) * K;
#pragma unroll
            for (int j = 0; j < PK; ++j) xr[i][j] = *reinterpret_cast<const h8_t *>(row + min((uint32_t)(j * 64 + lane), n_pieces - 1u) * 8u);
        }
    };
    uint32_t pass = first_pass;
    request_rows(pass, true);
    if constexpr (ORDERED) __builtin_amdgcn_sched_barrier(0);
    h8_t gv[PK];
    if constexpr (!ORDERED) {
#pragma unroll
        for (int j = 0; j < PK; ++j) gv[j] = *reinterpret_cast<const h8_t *>((gamma ? gamma : x_in) + min((uint32_t)(j * 64 + lane), n_pieces - 1u) * 8u);
    } else if (gamma) {
#pragma unroll
        for (int j = 0; j < PK; ++j) gv[j] = *reinterpret_cast<const h8_t *>(gamma + min((uint32_t)(j * 64 + lane), n_pieces - 1u) * 8u);
    } else {
#pragma unroll
        for (int j = 0; j < PK; ++j) gv[j] = h8_t{0, 0, 0, 0, 0, 0, 0, 0};
    }
    h8_t *const g_lds = reinterpret_cast<h8_t *>(smem + lds_rows_bytes<NT, NC, PK>());
    if (G_IN_LDS<PK> && !ORDERED) {
#pragma unroll
        for (int j = 0; j < PK; ++j) g_lds[j * 64 + lane] = gv[j];
    }
    if constexpr (ORDERED) __builtin_amdgcn_sched_barrier(0);
    // ---- block scales (block-quantised weights): [block][slot] f16 in LDS, fetched along the rows of the scale matrix, two at a
    // time where a row holds an even number (per lane and block of the operand they were 16 lines to a request). Past the last block
    // they are zero: an infinite scale would make NaN of the input's zeros there.
    _Float16 *const sc_lds = reinterpret_cast<_Float16 *>(smem + lds_rows_bytes<NT, NC, PK>() + (G_IN_LDS<PK> ? PK * 1024 : 0));
    constexpr int SLOTS = NT * 16, SC_STRIDE = scale_stride<NT>(), SC_LOADS = WB == 16 ? 1 : (SLOTS * PK * 8 + NTHREADS - 1) / NTHREADS;  // pairs per thread
    uint32_t sc_raw[SC_LOADS];
    auto scale_at = [&](int i, uint32_t &slot, uint32_t &kb2) __attribute__((always_inline)) -> bool {
        const uint32_t idx = (uint32_t)tid + (uint32_t)i * NTHREADS;
        slot = idx / (PK * 8), kb2 = idx % (PK * 8);
        return slot < (uint32_t)SLOTS;
    };
    if constexpr (WB != 16) {
#pragma unroll
        for (int i = 0; i < SC_LOADS; ++i) {
            uint32_t slot, kb2;
            int mat;
            bool valid;
            if (!scale_at(i, slot, kb2) || 2 * kb2 >= nkb) slot = 0, kb2 = 0;
            const uint32_t lrow = locate(slot_row(slot >> 4, slot & 15u, valid), mat);
            const __half *sp = pick3(mat, sp0, sp1, sp2) + (size_t)lrow * nkb + 2 * kb2;
            if (scale_pairs) {
                sc_raw[i] = fa_norm::load_global<uint32_t>(sp);
            } else {
                const uint32_t lo = fa_norm::load_global<unsigned short>(sp);
                sc_raw[i] = lo | ((uint32_t)fa_norm::load_global<unsigned short>(sp + (2 * kb2 + 1 < nkb ? 1 : 0)) << 16);
            }
        }
    }
    if constexpr (ORDERED) __builtin_amdgcn_sched_barrier(0);
    // ---- all weights of the workgroup. F16 (and SUMS, Q8_0): block kb of slot (t, n), features 8c .. 8c + 7. Block-quantised: 16
    // bytes per lane, half a block of one of two (Q8_0) or a block of four (Q4_0); the features that lane c holds for step s of such
    // a request follow from that, for the weights and for the input rows alike. SUMS wants a block in all lanes of a row: with Q4_0
    // that is 4 bytes to a lane, and a compute unit's address unit takes few lanes per cycle whatever they ask for. So the lanes
    // take 16 bytes along memory there (TURN) and the operand order is made in LDS when the weights are first used: Q4_0, 2 to 11
    // rows, 5120 x 3072 10.1 -> 9.2 us, row-major 12.6 -> 9.3; 3072 x 3072 6.4 -> 5.7, 7.9 -> 5.8; 2560 x 2048 7.7 -> 7.4. (Rows of
    // up to 1024 features are a request or two either way, row-major 1 to 5 % slower; F16 and the other block-quantised forms lose
    // 3 to 15 % by it, Q8_0 per-block sums 7 to 40 % for want of registers.)
    auto kb_of = [&](int i) __attribute__((always_inline)) -> uint32_t {
        return GB == 1 ? 16u * (uint32_t)(i >> 1) + 2u * (uint32_t)wave + (uint32_t)(i & 1) : GB == 2 ? 16u * (uint32_t)i + 2u * (uint32_t)wave : 32u * (uint32_t)i + 4u * (uint32_t)wave;
    };
    // the lane's row and block of a request: of its operand, and of what it fetches (blocked weights have a block of 16 rows side by side)
    const uint32_t lane_blk = GB == 1 ? 0u : GB == 2 ? (uint32_t)c >> 1 : (uint32_t)c;
    const uint32_t get_row = TURN && !canonical ? (uint32_t)lane >> 2 : (uint32_t)n, get_blk = TURN && !canonical ? (uint32_t)lane & 3u : lane_blk;
    // TURN: a KiB of LDS per wave, [block][row][16 bytes]
    unsigned char *const turn = smem + turn_at<WB, NT, NC, PK>() + wave * 1024;
    auto operand_order = [&](req_t &w) __attribute__((always_inline)) {
        if constexpr (TURN) {
            *reinterpret_cast<u4v_t *>(turn + get_blk * 256 + get_row * 16) = w;
#pragma unroll
            for (int b = 0; b < 4; ++b) w[b] = *reinterpret_cast<const uint32_t *>(turn + b * 256 + n * 16 + c * 4);
        }
    };
    req_t wv[NT][NA];
    const unsigned char *w_at[NT];  // block 0 of the lane's row in each tile, and how far apart blocks are
    uint32_t w_step[NT];
    // Weights are kept in the caches by kernels whose workgroups share them on an XCD, but for F16 rows of more than 1024 features in up to
    // two tiles, and block-quantised ones of more than 2048: the same kernels have launches that share nothing, which take 1.05 times as long
    // (o_proj of 3072 x 3072 F16, 5 rows 5.40 -> 5.67 us, of 2048 x 2048 16 rows 4.40 -> 4.61). 0.96 to 0.99 of the nontemporal loads' time in the mean
    // (250 launches of 9 to 64 rows): FusedQkv + KvPrepFused of 1152 x 896, 32 rows F16 4.33 -> 4.09, of 2560 x 2048, 24 rows Q8_0 6.14 -> 6.07, o_proj
    // of 2048 x 2048, 16 rows Q8_0 3.99 -> 3.80.
    constexpr bool SHARED = NT > 2 || (BESIDE && PK <= (WB == 16 ? 2 : 4));
    auto request_weights = [&](int t, int i) __attribute__((always_inline)) {
        const uint32_t kb = kb_of(i) + get_blk;
        const unsigned char *p = w_at[t] + (size_t)min(kb, nkb - 1u) * w_step[t];
        // (F16: zeros past the last block. The input is zero there, but an infinite weight read again would make NaN of it;
        // block-quantised weights are finite, and their scale is zero there.)
        if (WB == 16 && kb >= nkb) p = reinterpret_cast<const unsigned char *>(&zero_weights);
        wv[t][i % NA] = SHARED ? fa_norm::load_global<req_t>(p) : fa_norm::load_global_once<req_t>(p);
    };
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        bool valid;
        int mat;
        const uint32_t lrow = locate(slot_row((uint32_t)t, get_row, valid), mat);
        const uint32_t N = pick3(mat, rows0, rows1, rows1);
        // canonical (blocked by 32 features): (k % 32) + 32 * (row + (k / 32) * N); row-major: row * K + k
        const uint32_t in_block = GB == 1 ? (uint32_t)c * WB : GB == 2 ? ((uint32_t)c & 1u) * 16u : 0u;  // bytes
        w_at[t] = pick3(mat, w0, w1, w2) + (canonical ? (size_t)lrow * 32 : (size_t)lrow * K) * WB / 8 + in_block;
        w_step[t] = (canonical ? N * 32 : 32) * WB / 8;
        if constexpr (!RING) {
#pragma unroll
            for (int i = 0; i < NF; ++i) request_weights(t, i);
        }
    }
    if constexpr (RING) {
#pragma unroll
        for (int i = 0; i < NF; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) request_weights(t, i);
    }
    if constexpr (ORDERED) __builtin_amdgcn_sched_barrier(0);
    if (G_IN_LDS<PK> && ORDERED && gamma) {
#pragma unroll
        for (int j = 0; j < PK; ++j) g_lds[j * 64 + lane] = gv[j];
    }
    const float eps = a.eps, inv_k = a.inv_k, alpha = a.alpha, beta = a.beta;
    const __half *const residual = a.residual;
    const __half *const bias0 = a.bias[0], *const bias1 = a.bias[1], *const bias2 = a.bias[2];
    __half *const out0 = a.out[0], *const out1 = a.out[1], *const out2 = a.out[2];
    asm volatile("" ::"s"(residual), "s"(bias0), "s"(bias1), "s"(bias2), "s"(out0), "s"(out1), "s"(out2), "s"(eps), "s"(inv_k), "s"(alpha), "s"(beta));
    RopeDev r{};
    uint32_t block_shift = 32;  // log2 of the page size, 32 = not a power of two
    if constexpr (ROPE) {
        r = a.r, block_shift = a.block_shift;
        asm volatile("" ::"s"(r.cos_t), "s"(r.sin_t), "s"(r.block_table), "s"(r.n_kv_heads), "s"(r.position_offset), "s"(r.max_seq_len),
                     "s"(r.block_size), "s"(r.capacity), "s"(r.table_rows), "s"(r.apply), "s"(block_shift));
    }
    // ---- what the thread that stores slot (t, w_row) of input row w_col needs beside the sums; lanes of a store run along the
    // weight rows. Asked for ahead, from addresses that are valid whatever the slot.
    const uint32_t w_row = (uint32_t)tid & 15u, w_col = (uint32_t)tid >> 4;
    uint32_t s_row[NT];
    int s_mat[NT];
    bool s_ok[NT];
    _Float16 s_bias[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        s_row[t] = locate(slot_row((uint32_t)t, w_row, s_ok[t]), s_mat[t]);
        s_bias[t] = fa_norm::load_global<_Float16>(bias0 ? pick3(s_mat[t], bias0, bias1, bias2) + s_row[t] : x_in);
    }
    constexpr bool APART = REDUCE_APART<NT, NC, PK>;
    float *red = reinterpret_cast<float *>(smem + (APART ? NC * 16 * XROW : 0));  // [NW][NT][NC][16][17]; not APART: over the rows once they have been read

    while (true) {
        const uint32_t m0 = pass * PASS, cols = min(PASS, m_rows - m0), next = RING ? n_pass : pass + pass_step;
        if (gamma) {  // x * rsqrt(mean(x^2) + eps) * gamma in f32, rounded to f16; a wave holds whole rows
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                if (i > 0 && 8u * i >= cols) break;  // (uniform: no such rows in this pass. QKV of 18 .. 24 rows: 5 to 9 % less)
                float ss = 0.0f;
#pragma unroll
                for (int j = 0; j < PK; ++j) {
                    const float q = dot8_self(xr[i][j], 0.0f);
                    ss += (uint32_t)(j * 64 + lane) < n_pieces ? q : 0.0f;
                }
                const float inv_rms = fa_norm::inv_rms(fa_norm::wave_sum(ss), inv_k, eps);
#pragma unroll
                for (int j = 0; j < PK; ++j) xr[i][j] = fa_norm::scale8(xr[i][j], inv_rms, G_IN_LDS<PK> ? g_lds[j * 64 + lane] : gv[j]);
            }
        }
        // The longest rows: two chains of sums. Their error in units of 2^-24 of the sums' size, 12 to 64 rows of 2112 to 3072 features: F16 2.0, 2.4
        // with one; Q8_0 1.8 to 2.1 (one 2.1 to 2.4, the GEMM's tiles 2.0 to 2.3), Q4_0 1.8 to 2.1 (2.2 to 2.4, 3.0) for 0 to 1 % of the time.
        constexpr int CHAINS = PK > 4 && (WB == 16 || (RING && !SUMS)) ? 2 : 1;
        f4v_t d[NT][NC], d2[NT][NC];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int h = 0; h < NC; ++h) d[t][h] = d2[t][h] = f4v_t{0.0f, 0.0f, 0.0f, 0.0f};
        _Float16 s_res[NT], rc[NT], rs[NT];
        uint32_t r_pos = 0, r_blk = 0;
        if (!APART && pass != first_pass) __syncthreads();  // the sums have been read
#pragma unroll
        for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int j = 0; j < PK; ++j) {
                h8_t v = xr[i][j];
                if (j >= PK - 2 && (uint32_t)(j * 64 + lane) >= n_pieces) v = h8_t{0, 0, 0, 0, 0, 0, 0, 0};
                *reinterpret_cast<h8_t *>(smem + (wave + 8 * i) * XROW + (j * 64 + lane) * 16) = v;
            }
        if constexpr (WB != 16) {
            if (pass == first_pass) {
#pragma unroll
                for (int i = 0; i < SC_LOADS; ++i) {
                    uint32_t slot, kb2;
                    if (!scale_at(i, slot, kb2)) continue;
                    unsigned short *dst = reinterpret_cast<unsigned short *>(sc_lds) + 2 * kb2 * SC_STRIDE + slot;
                    dst[0] = 2 * kb2 < nkb ? (unsigned short)sc_raw[i] : (unsigned short)0;
                    dst[SC_STRIDE] = 2 * kb2 + 1 < nkb ? (unsigned short)(sc_raw[i] >> 16) : (unsigned short)0;
                }
            }
        }
        __syncthreads();
        // what this pass's write stage takes, then the next pass's rows
        if constexpr (ROPE) {
            r_pos = r.position_offset + m0 + min(w_col, cols - 1u);
            const uint32_t tp = min(r_pos, r.table_rows - 1u);  // stay inside the tables
            const uint32_t hmask = (1u << half_shift) - 1u;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const uint32_t hd = s_row[t] & (2u * hmask + 1u), tc = neox ? (hd & hmask) : (hd >> 1);
                rc[t] = fa_norm::load_global<_Float16>(r.cos_t + ((size_t)tp << half_shift) + tc);
                rs[t] = fa_norm::load_global<_Float16>(r.sin_t + ((size_t)tp << half_shift) + tc);
            }
            if (r.block_table) r_blk = (uint32_t)r.block_table[block_shift < 32 ? r_pos >> block_shift : r_pos / r.block_size];
        } else {
#pragma unroll
            for (int t = 0; t < NT; ++t)
                s_res[t] = fa_norm::load_global<_Float16>(
                    residual ? residual + (size_t)(m0 + min(w_col, cols - 1u)) * pick3(s_mat[t], rows0, rows1, rows1) + s_row[t] : x_in);
        }
        if constexpr (REST) {
            if (RING || pass == first_pass) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int i = NF; i < NQ; ++i) request_weights(t, i);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (!RING && next < n_pass) request_rows(next, false);
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            if (TURN && pass == first_pass) {
#pragma unroll
                for (int t = 0; t < NT; ++t) operand_order(wv[t][i % NA]);
            }
            const uint32_t kb = kb_of(i) + (TURN ? 0u : lane_blk);
            const unsigned char *xp = smem + n * XROW + kb * 64 + (GB == 1 || TURN ? c * 16 : GB == 2 ? (c & 1) * 32 : 0);
            const _Float16 *const scp = sc_lds + kb * SC_STRIDE + (SUMS ? c * 4 : n);
            req_t raw[NT];
            _Float16 sc[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                raw[t] = wv[t][i % NA];
                // (opaque: made f16 here in every pass, not ahead of the passes, where it would wait for the weights)
                if constexpr (WB != 16) asm volatile("" : "+v"(raw[t]));
                if constexpr (WIDE) sc[t] = scp[t * 16];
            }
#pragma unroll
            for (int st = 0; st < GB; ++st) {
                h8_t xb[NC];
#pragma unroll
                for (int h = 0; h < NC; ++h) xb[h] = *reinterpret_cast<const h8_t *>(xp + st * (TURN ? 64 : 16) + h * 16 * XROW);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    if constexpr (SUMS) {
                        typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
                        const h4_t s4 = *reinterpret_cast<const h4_t *>(scp + st * SC_STRIDE + t * 16);
                        const f4v_t z = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int h = 0; h < NC; ++h) {
                            raw_t w;
                            if constexpr (TURN) w = W::part(raw[t], st);
                            else w = raw[t];
                            const f4v_t blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(W::plain(w), xb[h], z, 0, 0, 0);
#pragma unroll
                            for (int q = 0; q < 4; ++q) d[t][h][q] += blk[q] * (float)s4[q];
                        }
                    } else {
                        const h8_t w = WB == 16 ? W::f16(W::part(raw[t], 0), (_Float16)1.0f) : W::f16(W::part(raw[t], st), sc[t]);
#pragma unroll
                        for (int h = 0; h < NC; ++h) {
                            f4v_t &sum = (GB == 1 ? i : st) % CHAINS ? d2[t][h] : d[t][h];
                            sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, xb[h], sum, 0, 0, 0);
                        }
                    }
                }
            }
            if constexpr (RING && !REST) {
                if (i + NA < NQ) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int t = 0; t < NT; ++t) request_weights(t, i + NA);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        if constexpr (CHAINS == 2) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int h = 0; h < NC; ++h) d[t][h] += d2[t][h];
        }
        if (!APART) __syncthreads();  // everyone has read the rows
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int h = 0; h < NC; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) red[(((wave * NT + t) * NC + h) * 16 + c * 4 + i) * 17 + n] = d[t][h][i];
        __syncthreads();
        if (w_col < NC * 16u) {
            const int h = (int)(w_col >> 4), cn = (int)(w_col & 15u);
            _Float16 y2[NT];
            float s2[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                float s = 0.0f;
#pragma unroll
                for (int w = 0; w < NW; ++w) s += red[(((w * NT + t) * NC + h) * 16 + w_row) * 17 + cn];
                s *= alpha;
                asm volatile("" : "+v"(s_bias[t]));  // (converted here, not ahead of the passes)
                if (bias0) s += (float)s_bias[t];
                s2[t] = s, y2[t] = (_Float16)s;
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if constexpr (ROPE) {
                    const uint32_t D = 2u << half_shift, half = 1u << half_shift;
                    // the mate: the same slot of the other tile, or 8 slots away in a tile of both halves (NeoX), or the neighbouring slot
                    const _Float16 y_adj = (_Float16)__shfl_xor((float)y2[t], NT % 2 == 1 && t == NT - 1 && neox ? 8 : 1, 64);
                    const _Float16 ym = (t ^ 1) < NT && neox ? y2[(t ^ 1) < NT ? t ^ 1 : 0] : y_adj;
                    if (!s_ok[t] || w_col >= cols) continue;
                    const uint32_t hd = s_row[t] & (D - 1u), head = s_row[t] >> (half_shift + 1);
                    const bool first = neox ? hd < half : (hd & 1u) == 0;
                    _Float16 y = y2[t];
                    if (s_mat[t] != 2 && r.apply) y = (_Float16)rope_one((float)y, (float)ym, (float)rc[t], (float)rs[t], first);
                    _Float16 *dst;
                    if (s_mat[t] == 0) {
                        dst = reinterpret_cast<_Float16 *>(out0) + ((size_t)head * m_rows + (m0 + w_col)) * D + hd;
                    } else {
                        if (r_pos >= r.capacity) continue;  // never outside the cache
                        const size_t crow = r.block_table ? (((size_t)r_blk * r.n_kv_heads + head) * r.block_size + (block_shift < 32 ? r_pos & (r.block_size - 1) : r_pos % r.block_size)) * D
                                                          : ((size_t)head * r.max_seq_len + r_pos) * D;
                        dst = reinterpret_cast<_Float16 *>(s_mat[t] == 1 ? out1 : out2) + crow + hd;
                    }
                    fa_norm::store_global(dst, y);
                } else {
                    if (!s_ok[t] || w_col >= cols) continue;
                    float s = s2[t];
                    if (residual) s += (float)s_res[t] * beta;
                    const uint32_t N = pick3(s_mat[t], rows0, rows1, rows1);
                    fa_norm::store_global(pick3(s_mat[t], out0, out1, out2) + (size_t)(m0 + w_col) * N + s_row[t], (_Float16)s);
                }
            }
        }
        if (RING || next >= n_pass) break;
        pass = next;
    }
}

template <int WB, int NT, int NC, int PK, bool ROPE, bool SUMS, bool FEW, bool EIGHTS = false, bool WALK = false>
fa_status launch_one(FaLaunchScope &scope, dim3 grid, const PanelDev &a) {
    constexpr int lds = lds_bytes<WB, NT, NC, PK, SUMS>();
    static std::atomic<uint64_t> allowed{0};  // devices this kernel's LDS size has been asked for on (the calls are idempotent)
    const uint64_t bit = 1ull << (scope.ctx->device & 63);
    if (!(allowed.load(std::memory_order_acquire) & bit)) {
        FA_HIP(hipFuncSetAttribute((const void *)panel_kernel<WB, NT, NC, PK, ROPE, SUMS, FEW, EIGHTS, WALK>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        allowed.fetch_or(bit, std::memory_order_release);
    }
    scope.launch(panel_kernel<WB, NT, NC, PK, ROPE, SUMS, FEW, EIGHTS, WALK>, grid, dim3(NTHREADS), lds, a);
    return FA_OK;
}
template <int WB, int NT, int NC, bool SUMS, bool FEW>
fa_status launch_pk(FaLaunchScope &scope, bool rope, uint32_t pk, dim3 grid, const PanelDev &a) {
    if (pk <= 2) return rope ? launch_one<WB, NT, NC, 2, true, SUMS, FEW>(scope, grid, a) : launch_one<WB, NT, NC, 2, false, SUMS, FEW>(scope, grid, a);
    if (NC == 2 || pk <= 4) return rope ? launch_one<WB, NT, NC, 4, true, SUMS, FEW>(scope, grid, a) : launch_one<WB, NT, NC, 4, false, SUMS, FEW>(scope, grid, a);
    return rope ? launch_one<WB, NT, 1, 6, true, SUMS, FEW>(scope, grid, a) : launch_one<WB, NT, 1, 6, false, SUMS, FEW>(scope, grid, a);  // (16 rows per pass: registers)
}
template <int WB, int NT, bool SUMS>
fa_status launch_eights(FaLaunchScope &scope, bool rope, uint32_t pk, dim3 grid, const PanelDev &a) {  // (rows of up to 2048 features)
    if (pk <= 2) return rope ? launch_one<WB, NT, 1, 2, true, SUMS, true, true>(scope, grid, a) : launch_one<WB, NT, 1, 2, false, SUMS, true, true>(scope, grid, a);
    return rope ? launch_one<WB, NT, 1, 4, true, SUMS, true, true>(scope, grid, a) : launch_one<WB, NT, 1, 4, false, SUMS, true, true>(scope, grid, a);
}
template <int WB, int NT>
fa_status launch_walk(FaLaunchScope &scope, bool rope, dim3 grid, const PanelDev &a) {  // (rows of more than 2048 features)
    return rope ? launch_one<WB, NT, 1, 6, true, false, false, false, true>(scope, grid, a) : launch_one<WB, NT, 1, 6, false, false, false, false, true>(scope, grid, a);
}
template <int WB>
fa_status launch(FaLaunchScope &scope, bool rope, bool sums, const Plan &plan, const PanelDev &a) {
    constexpr bool Q = WB != 16;  // (block-quantised weights have per-block sums wherever there are as few rows)
    const uint32_t nt = plan.nt, nc = plan.nc, pk = plan.pk;
    if (!has_kernel(Shape{a.total_rows, a.k_dim, a.m, (uint32_t)WB, a.canonical != 0, a.gamma != nullptr, rope}, plan))
        return fa_fail(FA_ERR_INVALID_OPERATION, "panel kernel: no form %d of %u tiles x %u groups for rows of %u features", (int)plan.form, nt, nc, a.k_dim);
    const dim3 grid = plan.form == WALK ? dim3(plan.grid_x, plan.grid_y) : dim3(plan.workgroups());
    if (a.m <= 8 && (!Q || sums)) return nt == 1 ? launch_pk<WB, 1, 1, Q, true>(scope, rope, pk, grid, a) : launch_pk<WB, 2, 1, Q, true>(scope, rope, pk, grid, a);
    if (plan.form == EIGHTS) {
        if constexpr (Q) {
            if (sums) return nt == 1 ? launch_eights<WB, 1, true>(scope, rope, pk, grid, a) : launch_eights<WB, 2, true>(scope, rope, pk, grid, a);
        }
        return nt == 1 ? launch_eights<WB, 1, false>(scope, rope, pk, grid, a) : launch_eights<WB, 2, false>(scope, rope, pk, grid, a);
    }
    if constexpr (Q) {
        if (sums) return nt == 1 ? launch_pk<WB, 1, 1, true, false>(scope, rope, pk, grid, a) : launch_pk<WB, 2, 1, true, false>(scope, rope, pk, grid, a);
    }
    if (plan.form == WALK && pk > 4) return nt == 1 ? launch_walk<WB, 1>(scope, rope, grid, a) : launch_walk<WB, 2>(scope, rope, grid, a);
    if (nt == 3 && pk <= 4) return rope ? launch_one<WB, 3, 1, 4, true, false, false>(scope, grid, a) : launch_one<WB, 3, 1, 4, false, false, false>(scope, grid, a);
    if (nt == 3) return rope ? launch_one<WB, 3, 1, 6, true, false, false>(scope, grid, a) : launch_one<WB, 3, 1, 6, false, false, false>(scope, grid, a);
    if (nt == 4) return rope ? launch_one<WB, 4, 1, 6, true, false, false>(scope, grid, a) : launch_one<WB, 4, 1, 6, false, false, false>(scope, grid, a);
    if constexpr (!Q) {
        if (nt == 5) return rope ? launch_one<WB, 5, 1, 6, true, false, false>(scope, grid, a) : launch_one<WB, 5, 1, 6, false, false, false>(scope, grid, a);
    }
    if (nt == 1) return nc == 1 ? launch_pk<WB, 1, 1, false, false>(scope, rope, pk, grid, a) : launch_pk<WB, 1, 2, false, false>(scope, rope, pk, grid, a);
    return nc == 1 ? launch_pk<WB, 2, 1, false, false>(scope, rope, pk, grid, a) : launch_pk<WB, 2, 2, false, false>(scope, rope, pk, grid, a);
}

}  // namespace fa_panel
