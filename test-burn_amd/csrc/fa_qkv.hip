// FusedQkv: RMSNorm(input) -> Q, K and V projections in one launch -> three token-major outputs, F16 weights.
// Reference: src/metals/gemv/qkv_step.rs:14-120,220-460 (step, arguments, dispatch), src/metals/gemv/qkv_project.metal
// (projection, reduce, bias + write), src/metals/rmsnorm/rmsnorm.metal:17-96 (inv_rms), weight layouts
// src/compound/stages/layout.rs:79-100.
//
// The reference gives every output row a 32-lane warp and re-reads the input per row. Here the step is what it is
// at decode, a weight stream (HBM-bound: every weight is read once per launch, the input is a few KB):
//   * the rows of W_q, W_k, W_v are treated as one list and dealt evenly to a multiple of the CU count of
//     workgroups (not in 16-row quanta: 5120 rows over 256 CUs are 512 workgroups of 10), so that every CU
//     requests the same number of bytes;
//   * a workgroup walks its rows in tiles of 16; a tile times 32 input features is one 1 KiB load per wave in the
//     blocked ("canonical") layout, and one v_mfma_f32_16x16x32_f16 with the (<= 16) input rows as the other
//     operand - the matrix unit is used for its shape, not its rate: columns past m are zero;
//   * the 8 waves split the feature blocks of a tile; their 16 x 16 partial results are summed through LDS in a
//     fixed order, the bias is added and the row is rounded to f16 once, as the reference does.
// The normalised input is rounded to f16 before the products (qkv_project.metal:66-67), f32 accumulation.
// Q8_0 weights (src/metals/policies/policy_q8.metal: int8 values, one f16 scale per 32 weights of a row, separate
// buffers) take the same route at half the bytes: 8 bytes per lane and block, converted to f16 exactly, one matrix
// instruction per 32-weight block whose row sums are multiplied by the block's scales (staged in LDS) and added up.
// Q4_0 weights (policy_q4_0.metal: nibble - 8, adjacent pairs per byte, the same scales) at a quarter: 4 bytes per lane.
//
// The same kernel with one matrix, no norm and the write stage's alpha / bias / beta * residual is the m = 1 path of
// the MatMul op (src/metals/matmul.rs:190-239 -> GemvV2, write stage src/metals/gemv/stages.rs:200-224): the o_proj
// consumer of the attention output.
#include "fa_internal.h"
#include "fa_norm.h"
#include "fa_panel.h"
#include "fa_qkv_rope.h"
#include "fa_quant.h"
#include <algorithm>
#include <atomic>
#include <type_traits>

namespace {

constexpr int QKV_NT = 512, QKV_NW = QKV_NT / 64;
constexpr int QKV_UNITS = 8;  // feature blocks per batch of requests; a wave keeps two batches in flight
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4v_t __attribute__((ext_vector_type(4)));
typedef unsigned int u2v_t __attribute__((ext_vector_type(2)));

struct QkvDev {
    const __half *w[3];     // W_q, W_k, W_v
    const __half *bias[3];  // nullable as a set
    __half *out[3];         // [m, rows[i]]
    uint32_t rows[3];       // n_dim, n_kv, n_kv
    const __half *x;        // [m, k_dim]
    const __half *gamma;    // nullable: no RMSNorm
    uint32_t k_dim, m, cols_per_pass, rows_per_wg, x_stride /* bytes of an input row in LDS */, canonical;
    float eps;
    // MatMul form (one matrix): out = f16(alpha * sum + bias + beta * residual)
    const __half *residual;  // nullable; [m, rows[0]]
    float alpha, beta;
    // Q8_0 weights: w[i] point at int8 values (same two layouts, in elements), scales[i] at f16 [rows, k_dim / 32]
    const __half *scales[3];
    uint32_t rcp_nkb;  // floor(2^32 / (k_dim / 32)) + 1: exact quotients of a workgroup's scale indices (below 2^16)
};

// One of three values by matrix index. (Taken by value on purpose: `mat == 0 ? x0 : mat == 1 ? x1 : x2` written out on
// variables is a conditional LVALUE - the compiler selects an address and loads through it, per lane, which keeps the three
// in memory: launch arguments were fetched with a vector load from the argument block, locals went to scratch.)
template <typename T>
__device__ __forceinline__ T pick3(int mat, T x0, T x1, T x2) {
    return mat == 0 ? x0 : mat == 1 ? x1 : x2;
}

// WB: bits per weight - 16 (f16), 8 (Q8_0) or 4 (Q4_0)
template <int WB>
__global__ void __launch_bounds__(QKV_NT, 2) fused_qkv_kernel(QkvDev a_by_value) {
    constexpr bool Q8 = WB != 16;  // block-quantised: integer weights + one f16 scale per 32 of a row
    constexpr bool Q4 = WB == 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // The arguments are read straight from the launch's argument block (the struct is its only member) into locals, those
    // that the first weight request needs in one trip through the scalar cache. As a by-value struct the per-matrix
    // pointers were fetched where a row's matrix was known - `mat == 0 ? a.w[0] : ...` became a per-lane VECTOR load
    // from the argument block, with a wait for it (and for the input row requested before it) ahead of the first
    // weight request: a trip to memory before the stream could start, and another per tile for bias and output.
    static_assert(std::is_trivially_copyable<QkvDev>::value, "read as raw bytes from the argument block, where it is the first member");
    const QkvDev &a = *(const QkvDev *)__builtin_amdgcn_kernarg_segment_ptr();
    (void)a_by_value;
    const unsigned char *const w0 = reinterpret_cast<const unsigned char *>(a.w[0]), *const w1 = reinterpret_cast<const unsigned char *>(a.w[1]),
                        *const w2 = reinterpret_cast<const unsigned char *>(a.w[2]);
    const uint32_t rows0 = a.rows[0], rows1 = a.rows[1], rows2 = a.rows[2];
    const __half *const x_in = a.x, *const gamma = a.gamma;
    const uint32_t K = a.k_dim, m_rows = a.m, cols_per_pass = a.cols_per_pass, rows_per_wg = a.rows_per_wg, x_stride = a.x_stride;
    const uint32_t canonical_u = a.canonical;
    asm volatile("" ::"s"(w0), "s"(w1), "s"(w2), "s"(rows0), "s"(rows1), "s"(rows2), "s"(x_in), "s"(gamma), "s"(K), "s"(m_rows), "s"(cols_per_pass),
                 "s"(rows_per_wg), "s"(x_stride), "s"(canonical_u));
    const bool canonical = canonical_u != 0;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, c = lane >> 4;
    const uint32_t nkb = K / 32;
    const uint32_t total_rows = rows0 + rows1 + rows2;
    const uint32_t row_begin = blockIdx.x * rows_per_wg;
    const uint32_t row_end = min(total_rows, row_begin + rows_per_wg);
    if (row_begin >= row_end) return;
    const uint32_t n_tiles = (row_end - row_begin + 15) / 16;
    const uint32_t m0 = blockIdx.y * cols_per_pass, cols = min(cols_per_pass, m_rows - m0);
    unsigned char *x_lds = smem;
    float *red = reinterpret_cast<float *>(smem + (size_t)cols_per_pass * x_stride);  // [QKV_NW][16][17], and scratch
    // Q8: the block scales of this workgroup's rows, [tile][feature block][16 rows] f16
    _Float16 *sc_lds = reinterpret_cast<_Float16 *>(red + QKV_NW * 16 * 17);

    // Where a row of the concatenated list lives: matrix, row inside it, the matrix's row count.
    auto locate = [&](uint32_t gr, int &mat, uint32_t &lrow) __attribute__((always_inline)) {
        mat = 0, lrow = gr;
        if (lrow >= rows0) {
            lrow -= rows0, mat = 1;
            if (lrow >= rows1) lrow -= rows1, mat = 2;
        }
    };
    // Weight operand of (tile, feature block kb): lane (n, c) holds features 8c..8c+7 of the block for row n of the
    // tile (consecutive lanes 64 bytes apart; requesting in address order, four lanes per row, and moving the words
    // into place with LDS permutes was slower: 10.6 us against 9.5 on 31.5 MB of weights).
    // Per tile a lane keeps the address of its block 0 and its stride from block to block.
    // (Q8: the same element indices, one byte per element.)
    // (Q4: two elements per byte, element 2i in the low nibble of byte i.)
    typedef typename std::conditional<Q4, uint32_t, typename std::conditional<Q8, u2v_t, h8_t>::type>::type wreg_t;
    auto tile_base = [&](uint32_t tile, const unsigned char *&p0, size_t &kb_stride, bool &ok) __attribute__((always_inline)) {
        const uint32_t gr = row_begin + tile * 16 + n;
        ok = gr < row_end;
        int mat;
        uint32_t lrow;
        locate(ok ? gr : row_begin, mat, lrow);
        const unsigned char *base = pick3(mat, w0, w1, w2);
        const uint32_t N = pick3(mat, rows0, rows1, rows1);
        // canonical (blocked by 32 features): (k % 32) + 32 * (row + (k / 32) * N); row-major: row * K + k
        p0 = base + (canonical ? (size_t)lrow * 32 + c * 8 : (size_t)lrow * K + c * 8) * WB / 8;
        kb_stride = (canonical ? (size_t)N * 32 : 32) * WB / 8;
    };

    // A wave takes the feature blocks kb = wave, wave + 8, ... of every tile, in batches of QKV_UNITS; two batches
    // are in flight. The first two are requested before anything else: they do not depend on the input.
    const uint32_t per_tile = (nkb + QKV_NW - 1) / QKV_NW;                // blocks of a tile per wave (upper bound)
    const uint32_t bpt = (per_tile + QKV_UNITS - 1) / QKV_UNITS;          // batches per tile
    const uint32_t n_batches = n_tiles * bpt;
    wreg_t wbuf[2][QKV_UNITS];
    // `every`: all QKV_UNITS requests are made, one past the row's last block re-reads the last block (the first batch of
    // a workgroup is asked for this way: from 2048 features on none of its blocks is past the end, and with a fixed
    // number of requests behind the input row's the compiler can wait for that row alone - with a wave-dependent
    // number it waited for every weight of the first two batches before the normalisation could start).
    auto request = [&](wreg_t(&buf)[QKV_UNITS], uint32_t batch, bool every) __attribute__((always_inline)) {
        const uint32_t tile = batch / bpt, j0 = (batch % bpt) * QKV_UNITS;
        const unsigned char *p0;
        size_t kb_stride;
        bool ok;
        tile_base(tile, p0, kb_stride, ok);
#pragma unroll
        for (int i = 0; i < QKV_UNITS; ++i) {
            const uint32_t kb = (uint32_t)wave + (j0 + i) * QKV_NW;
            // weights are read once per launch: non-temporal, so that they do not push everything else out of the L2.
            // Every lane loads (a lane whose row is past the workgroup's last reads the first row's block: its sums
            // are never written), and a block past the row's last is skipped by the whole wave and never consumed. No
            // lane-dependent branch and no zero to merge with: with `(ok && kb < nkb) ? load : 0` the compiler
            // moved a loaded register right behind every other request - a wait for ALL requests so far, one trip to
            // memory per pair of requests.
            if (every) buf[i] = __builtin_nontemporal_load(reinterpret_cast<const wreg_t *>(p0 + (size_t)min(kb, nkb - 1) * kb_stride));
            else if (kb < nkb) buf[i] = __builtin_nontemporal_load(reinterpret_cast<const wreg_t *>(p0 + (size_t)kb * kb_stride));
        }
    };
    // The first input row is requested before the weights (a CU's vector loads return in request order), then the
    // first two batches, which do not depend on the input.
    constexpr int XPRE = 2;  // 16-byte pieces per thread: rows of up to 8192 features
    h8_t x0[XPRE];
#pragma unroll
    for (int j = 0; j < XPRE; ++j) {
        const uint32_t k8 = tid + j * QKV_NT;
        const h8_t z = {0, 0, 0, 0, 0, 0, 0, 0};
        x0[j] = k8 < K / 8 ? *reinterpret_cast<const h8_t *>(x_in + (size_t)m0 * K + k8 * 8) : z;
    }
    // ... and with it this thread's pieces of the norm's weights (of the input row again when there is no norm, so that
    // the number of requests does not depend on it): requested behind the weights they would arrive behind them.
    h8_t g0[XPRE];
#pragma unroll
    for (int j = 0; j < XPRE; ++j) {
        const uint32_t k8 = tid + j * QKV_NT;
        const h8_t z = {0, 0, 0, 0, 0, 0, 0, 0};
        g0[j] = k8 < K / 8 ? *reinterpret_cast<const h8_t *>((gamma ? gamma : x_in) + k8 * 8) : z;
    }
    // Q8: the block scales of this workgroup's rows (scales[row][kb] f16, row-major,
    // tests/gemv_v2_parity.rs:100-102); they go to LDS as [tile][kb][row].
    constexpr int SPRE = 4;
    _Float16 sc0[SPRE];
    const __half *const sc_p0 = Q8 ? a.scales[0] : nullptr, *const sc_p1 = Q8 ? a.scales[1] : nullptr, *const sc_p2 = Q8 ? a.scales[2] : nullptr;
    const uint32_t rcp_nkb = Q8 ? a.rcp_nkb : 0u;
    if (Q8) asm volatile("" ::"s"(sc_p0), "s"(sc_p1), "s"(sc_p2), "s"(rcp_nkb));
    // (index / nkb as a product: four divisions per thread stood between the launch's entry and its first weight request)
    auto div_nkb = [&](uint32_t idx) __attribute__((always_inline)) -> uint32_t { return nkb == 1 ? idx : __umulhi(idx, rcp_nkb); };
    const uint32_t n_scales = Q8 ? n_tiles * 16 * nkb : 0u;
    auto scale_of = [&](uint32_t idx) __attribute__((always_inline)) -> _Float16 {
        const uint32_t tr = div_nkb(idx), kb = idx - tr * nkb;  // tr = tile * 16 + row
        const uint32_t gr = row_begin + tr;
        if (gr >= row_end) return (_Float16)0.0f;
        int mat;
        uint32_t lrow;
        locate(gr, mat, lrow);
        const __half *sp = pick3(mat, sc_p0, sc_p1, sc_p2);
        return *reinterpret_cast<const _Float16 *>(sp + (size_t)lrow * nkb + kb);
    };
    request(wbuf[0], 0, true);
    // (the scales behind the first batch: their addresses take a few hundred instructions, which the first weight
    // requests should not wait for; they are needed when that batch is consumed)
    if (Q8) {
#pragma unroll
        for (int j = 0; j < SPRE; ++j) {
            const uint32_t idx = tid + j * QKV_NT;
            sc0[j] = idx < n_scales ? scale_of(idx) : (_Float16)0.0f;
        }
    }
    if (n_batches > 1) request(wbuf[1], 1, false);
    // (what the normalisation and the write stage take, while the first requests are on their way)
    const __half *const residual = a.residual;
    const __half *const bias0 = a.bias[0], *const bias1 = a.bias[1], *const bias2 = a.bias[2];
    __half *const out0 = a.out[0], *const out1 = a.out[1], *const out2 = a.out[2];
    const float eps = a.eps, alpha = a.alpha, beta = a.beta;
    asm volatile("" ::"s"(residual), "s"(bias0), "s"(bias1), "s"(bias2), "s"(out0), "s"(out1), "s"(out2), "s"(eps), "s"(alpha), "s"(beta));
    // The thread that will store (row, column) of the first tile asks for its bias and residual here, behind the weights: asked
    // for where they are added, after the last sum, they put another trip to memory between the products and the store. (Every
    // lane loads, from an address that is valid whatever its slot: no branch around a load.)
    const uint32_t w_row = ((uint32_t)tid >> 4) & 15u, w_col = (uint32_t)tid & 15u;
    _Float16 pre_bias, pre_res;
    {
        int mat;
        uint32_t lrow;
        locate(min(row_begin + w_row, row_end - 1u), mat, lrow);
        const __half *pb = bias0 ? pick3(mat, bias0, bias1, bias2) + lrow : x_in;
        const uint32_t N = pick3(mat, rows0, rows1, rows1);
        const __half *pr = residual ? residual + (size_t)(m0 + min(w_col, cols - 1u)) * N + lrow : x_in;
        pre_bias = *reinterpret_cast<const _Float16 *>(pb), pre_res = *reinterpret_cast<const _Float16 *>(pr);
    }

    // Input rows of this pass into LDS, normalised: x * rsqrt(mean(x^2) + eps) * gamma in f32, rounded to f16.
    // Four rows or more: a wave takes whole rows (row r by wave r % 8) and needs no workgroup barrier for the sum of
    // squares, so the rows are staged side by side instead of one after the other with two barriers each.
    const bool rows_by_wave = cols >= 4;  // measured on 5120 x 3072: 2 rows 9.2 us row after row, 10.4 by wave; 4 rows 11.3 / 10.5; 8 rows 15.7 / 11.1
    if (rows_by_wave) {
        for (uint32_t r = wave; r < cols; r += QKV_NW) {
            const __half *xr = x_in + (size_t)(m0 + r) * K;
            unsigned char *dst = x_lds + (size_t)r * x_stride;
            float ss = 0.0f;
            for (uint32_t k8 = lane; k8 < K / 8; k8 += 64) {
                const h8_t v = *reinterpret_cast<const h8_t *>(xr + k8 * 8);
                *reinterpret_cast<h8_t *>(dst + k8 * 16) = v;
#pragma unroll
                for (int i = 0; i < 8; ++i) ss += (float)v[i] * (float)v[i];
            }
            if (gamma) {
                const float inv_rms = rsqrtf(fa_norm::wave_sum(ss) / (float)K + eps);
                for (uint32_t k8 = lane; k8 < K / 8; k8 += 64) {  // each lane rewrites what it wrote
                    h8_t v = *reinterpret_cast<const h8_t *>(dst + k8 * 16);
                    const h8_t g = *reinterpret_cast<const h8_t *>(gamma + k8 * 8);
#pragma unroll
                    for (int i = 0; i < 8; ++i) v[i] = (_Float16)(((float)v[i] * inv_rms) * (float)g[i]);
                    *reinterpret_cast<h8_t *>(dst + k8 * 16) = v;
                }
            }
        }
    }
    for (uint32_t r = 0; r < (rows_by_wave ? 0u : cols); ++r) {
        const __half *xr = x_in + (size_t)(m0 + r) * K;
        unsigned char *dst = x_lds + (size_t)r * x_stride;
        float ss = 0.0f;
        for (uint32_t k8 = tid, j = 0; k8 < K / 8; k8 += QKV_NT, ++j) {
            h8_t v;
            if (r == 0 && j < (uint32_t)XPRE) v = j == 0 ? x0[0] : x0[1];
            else v = *reinterpret_cast<const h8_t *>(xr + k8 * 8);
            *reinterpret_cast<h8_t *>(dst + k8 * 16) = v;
#pragma unroll
            for (int i = 0; i < 8; ++i) ss += (float)v[i] * (float)v[i];
        }
        if (gamma) {
            ss = fa_norm::wave_sum(ss);
            if (lane == 0) red[wave] = ss;
            __syncthreads();
            float tot = 0.0f;
#pragma unroll
            for (int w = 0; w < QKV_NW; ++w) tot += red[w];
            const float inv_rms = rsqrtf(tot / (float)K + eps);
            for (uint32_t k8 = tid, j = 0; k8 < K / 8; k8 += QKV_NT, ++j) {  // each thread rewrites what it wrote
                h8_t v;
                if (r == 0 && j < (uint32_t)XPRE) v = j == 0 ? x0[0] : x0[1];
                else v = *reinterpret_cast<const h8_t *>(dst + k8 * 16);
                h8_t g;
                if (j < (uint32_t)XPRE) g = j == 0 ? g0[0] : g0[1];
                else g = *reinterpret_cast<const h8_t *>(gamma + k8 * 8);
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = (_Float16)(((float)v[i] * inv_rms) * (float)g[i]);
                *reinterpret_cast<h8_t *>(dst + k8 * 16) = v;
            }
            if (r + 1 < cols) __syncthreads();  // `red` is reused by the next row
        }
    }
    if (Q8) {
        for (uint32_t idx = tid, j = 0; idx < n_scales; idx += QKV_NT, ++j) {
            const _Float16 v = j < (uint32_t)SPRE ? (j == 0 ? sc0[0] : j == 1 ? sc0[1] : j == 2 ? sc0[2] : sc0[3]) : scale_of(idx);
            const uint32_t tr = div_nkb(idx), kb = idx - tr * nkb;
            sc_lds[((size_t)(tr >> 4) * nkb + kb) * 16 + (tr & 15)] = v;
        }
    }
    __syncthreads();

    // Sums the 8 waves' partial results of tile t in wave order, adds the bias, rounds once, stores token-major.
    auto finish_tile = [&](uint32_t t, const f4v_t &mine) __attribute__((always_inline)) {
        if (t) __syncthreads();  // `red` may still be read for the previous tile
#pragma unroll
        for (int i = 0; i < 4; ++i) red[((size_t)wave * 16 + c * 4 + i) * 17 + n] = mine[i];
        __syncthreads();
        if (tid < 256) {
            const int row = tid >> 4, col = tid & 15;
            const uint32_t gr = row_begin + t * 16 + row;
            if (gr < row_end && (uint32_t)col < cols) {
                float s = 0.0f;
#pragma unroll
                for (int w = 0; w < QKV_NW; ++w) s += red[((size_t)w * 16 + row) * 17 + col];
                int mat;
                uint32_t lrow;
                locate(gr, mat, lrow);
                const __half *bias = pick3(mat, bias0, bias1, bias2);
                __half *out = pick3(mat, out0, out1, out2);
                const uint32_t N = pick3(mat, rows0, rows1, rows1);
                s *= alpha;
                if (bias) s += t ? __half2float(bias[lrow]) : (float)pre_bias;
                if (residual) s += (t ? __half2float(residual[(size_t)(m0 + col) * N + lrow]) : (float)pre_res) * beta;
                out[(size_t)(m0 + col) * N + lrow] = __float2half(s);
            }
        }
    };

    // Stream: d = 16 rows of the current tile x 16 input rows, this wave's share of the feature blocks. Batches run
    // tile after tile and every wave sees the same sequence, so a tile is finished when its last batch is consumed.
    f4v_t d = {0.0f, 0.0f, 0.0f, 0.0f};
    const bool col_ok = (uint32_t)n < cols;
    const unsigned char *x_lane = x_lds + (size_t)(col_ok ? n : 0) * x_stride + c * 16;
    auto consume = [&](const wreg_t(&buf)[QKV_UNITS], uint32_t batch) __attribute__((always_inline)) {
        const uint32_t tile = batch / bpt, j0 = (batch % bpt) * QKV_UNITS;
#pragma unroll
        for (int i = 0; i < QKV_UNITS; ++i) {
            const uint32_t kb = (uint32_t)wave + (j0 + i) * QKV_NW;
            if (kb >= nkb) break;  // wave-uniform
            h8_t xb = *reinterpret_cast<const h8_t *>(x_lane + kb * 64);
            if (!col_ok) xb = h8_t{0, 0, 0, 0, 0, 0, 0, 0};
            if constexpr (Q8) {
                // 8 int8 weights -> f16 (exact); one MFMA covers exactly one 32-weight block, whose sums are scaled
                // per row (lane (n, c) of the result holds rows 4c..4c+3) and then accumulated
                h8_t wv;
                if constexpr (Q4) wv = fa_quant::q4_to_f16(buf[i]);
                else wv = fa_quant::q8_to_f16(buf[i][0], buf[i][1]);
                const f4v_t z = {0.0f, 0.0f, 0.0f, 0.0f};
                const f4v_t blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv, xb, z, 0, 0, 0);
                typedef _Float16 h4v_t __attribute__((ext_vector_type(4)));
                const h4v_t sc = *reinterpret_cast<const h4v_t *>(sc_lds + ((size_t)tile * nkb + kb) * 16 + c * 4);
#pragma unroll
                for (int q = 0; q < 4; ++q) d[q] += blk[q] * (float)sc[q];
            } else {
                d = __builtin_amdgcn_mfma_f32_16x16x32_f16(buf[i], xb, d, 0, 0, 0);
            }
        }
        if ((batch + 1) % bpt == 0) {
            finish_tile(tile, d);
            d = f4v_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
    };
    for (uint32_t b = 0; b < n_batches; b += 2) {
        consume(wbuf[0], b);
        if (b + 2 < n_batches) request(wbuf[0], b + 2, false);
        if (b + 1 < n_batches) {
            consume(wbuf[1], b + 1);
            if (b + 3 < n_batches) request(wbuf[1], b + 3, false);
        }
    }
}

}  // namespace

static fa_panel::Shape panel_shape(const FusedQkvLaunch &l, bool rope) {
    return {l.n_dim + 2 * l.n_kv, l.k_dim, l.m, (uint32_t)l.weight_bits, l.canonical, l.gamma != nullptr, rope};
}

// Whether a FusedQkv / MatMul launch goes to the panel kernel: rows of up to 3072 features, from two input rows (four layers of the
// Llama-3.2-3B block with 2 / 4 / 8 / 11 rows: 113 / 113 / 115 / 117 us against 120 / 128 / 137 / 155 with the kernel for up to 16
// rows). Up to 32 rows whose weight rows fit one round of workgroups always (a default chunk is one launch). Beyond, up to as many as
// it is measured to beat the tile kernels with where the weight rows suit it - later where those need the normalisation's launch in
// front (Qwen2.5-0.5B: 384 rows, both 31.8 us per layer; its o_proj alone, F16: 128 rows 4.2 against 5.0 us, 256 rows 5.3 against
// 5.1; block-quantised as long as each pass has a workgroup of its own, two to a compute unit, 239 rows of 896 x 192 Q4_0 3.8 against
// 5.2, 314 rows of 512 x 128 Q8_0 3.7 against 4.4, 228 rows of 640 x 960 Q4_0 4.5 against 4.8, 265 rows of 896 x 704 Q8_0 row-major
// both 5.2, 30 launches 0.85 in the mean and 1.13 at worst; of 256 features only one to a compute unit, 438 rows of 256 x 576 take
// 1.17 times as long as the tiles) - unless the GEMM is a tenth ahead by
// estimate: many weight rows are many passes of the input rows here, or rounds of workgroups. A launch takes the weight stream, and
// for each pass that a compute unit has one after the other the input rows of that pass, fetched and multiplied and, with a gamma,
// normalised (fitted to walks over passes, of launches of 12 to 416 rows over 512 to 3072 features and 512 to 10240 weight rows; a
// workgroup for each pass, where there is one, takes less than the estimate says, so that what stays would stay). us, here and as a GEMM:
// 2048 x 10240 32 rows 16.6, 12.4, 100 rows 44.5, 17.6; 2048 x 2560 64 rows 8.2, 11.0, 100 rows 12.8, 11.1; 1024 x 6144 100 rows 13.2, 8.8. An
// explicit GEMM threshold (fa_set_gemm_min_m) wins.
bool fa_qkv_rows32_takes(const fa_ctx *ctx, const FusedQkvLaunch &l) {
    constexpr uint32_t PANEL_MIN_M_DEFAULT = 2;
    auto aligned16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    const uint32_t min_m = ctx->qkv_rows32_min_m ? ctx->qkv_rows32_min_m : PANEL_MIN_M_DEFAULT;
    const bool f16 = l.weight_bits == 16;
    const uint32_t max_m = l.k_dim <= 1024 ? (l.gamma ? 416u : f16 ? 192u : 512u) : l.k_dim <= 2048 ? 128u : 64u;
    if (min_m > 32 || l.m < min_m || l.m > max_m || l.k_dim > 3072 || l.k_dim % 32 != 0) return false;
    if (ctx->gemm_min_m && (l.weight_bits != 16 || l.m >= ctx->gemm_min_m)) return false;
    if (!aligned16(l.x) || !aligned16(l.w[0]) || !aligned16(l.w[1]) || !aligned16(l.w[2]) || !aligned16(l.gamma)) return false;
    if (l.m < FA_GEMM_MIN_M_DEFAULT) return true;
    const uint32_t n_cus = ctx->n_cus > 0 ? (uint32_t)ctx->n_cus : 256u;
    // (the write stage must not decide: a fused op takes the route of its two ops)
    const fa_panel::Shape shape = panel_shape(l, false);
    const bool tiles_fit = fa_gemm_tiles_fit(l);  // (where they don't, the GEMM is a divided one of three launches: 1.5 to 4 times as long)
    if (l.k_dim > 2048 && l.m > 16) {
        // A workgroup for each pass: 0.69 to 0.97 of the tiles' time, but for F16 row-major weights in five tiles (1.09 to 1.36, 16 launches) and
        // block-quantised ones, which are made f16 for each pass, in four tiles: up to 2560 features Q4_0 1.09, Q8_0 1.06 and with a gamma 0.95;
        // longer Q4_0 1.04 and with a gamma 0.97, Q8_0 0.93 and 0.90 (75 launches in all).
        const fa_panel::Plan b = fa_panel::panel_plan(shape, n_cus);
        const bool q8 = l.weight_bits == 8;
        if (b.form == fa_panel::BESIDE)
            return !tiles_fit || (f16 ? l.canonical || b.nt < 5 : b.nt < 4 || (l.k_dim <= 2560 ? q8 && l.gamma != nullptr : q8 || l.gamma != nullptr));
        if (!f16 && tiles_fit && b.grid_y < b.n_pass) return false;  // (walking over passes: 1.2 to 3 times the tiles' time, 200 launches)
    }
    const fa_panel::Plan p = fa_panel::walk_plan(shape, n_cus);
    if (l.m <= 32 && p.rounds == 1) return true;
    if (l.k_dim > 2048 && tiles_fit && p.rounds > 1) return false;  // (1.06 to 3.2 times the tiles' time, 50 launches)
    if (!l.gamma && l.m > 192 && (uint64_t)ceil_div_u32(l.n_dim + 2 * l.n_kv, 16) * p.n_pass > (l.k_dim >= 512 ? 2 : 1) * n_cus) return false;
    // Block-quantised with a norm: where 32 input rows x 32 weight rows are more than a piece per compute unit, a second pass costs 3 us
    // and more, which the estimate below does not see of few features: 195 rows, 512 x 2112 Q4_0 12.0 us, 8.4 with the norm's launch and
    // the tiles; 391 rows, 640 x 1344 Q8_0 12.1, 9.2; 124 rows, 1280 x 2112 Q8_0 14.4, 9.3; 375 rows, 768 x 1664 13.8, 9.6; 248 rows,
    // 896 x 1664 Q4_0 9.65, 8.5; just below the line 192 rows, 512 x 1344 6.2, 7.2. (100 launches of 768 to 1024 features between one
    // piece and two: 0.71 to 0.975 of the panel kernel's time, 0.87 in the mean; 180 of 256 to 2048 features below the line: 1.09 to 1.32.)
    if (!f16 && l.gamma && l.m > 32 && p.nc == 2 && tiles_fit && (uint64_t)ceil_div_u32(l.n_dim + 2 * l.n_kv, 32) * p.n_pass > n_cus) return false;
    // passes of a compute unit (with two workgroups on it they share its way to L2)
    const float passes = p.pk > 2 ? (float)(p.rounds * ceil_div_u32(p.n_pass, p.grid_y)) : std::max(1.0f, (float)(p.grid_x * p.n_pass) / (float)n_cus);
    const float k = (float)l.k_dim, mb = k * (float)(l.n_dim + 2 * l.n_kv) * (f16 ? 2.0f : l.weight_bits == 8 ? 1.0625f : 0.5625f) * 1e-6f;
    const float per_pass = (float)p.nc * k / 1024.0f * (f16 ? (l.gamma ? 1.23f : 0.78f) : l.gamma ? 1.47f : 0.94f);
    return fa_gemm_estimate_us(ctx, l) >= 0.9f * (2.5f + (f16 ? 0.09f : 0.115f) * mb + passes * per_pass);
}

static fa_status launch_panel(fa_ctx *ctx, const FusedQkvLaunch &l, const QkvRopeLaunch *rope) {
    fa_panel::PanelDev a;
    memset(&a, 0, sizeof(a));
    for (int i = 0; i < 3; ++i)
        a.w[i] = reinterpret_cast<const unsigned char *>(l.w[i]), a.scales[i] = l.scales[i], a.bias[i] = l.bias[i], a.out[i] = l.out[i];
    a.rows0 = l.n_dim, a.rows1 = l.n_kv, a.total_rows = l.n_dim + 2 * l.n_kv;
    a.x = l.x, a.gamma = l.gamma, a.residual = l.residual, a.k_dim = l.k_dim, a.m = l.m, a.canonical = l.canonical ? 1u : 0u;
    a.eps = l.eps, a.inv_k = 1.0f / (float)l.k_dim, a.alpha = l.alpha, a.beta = l.beta;
    if (rope) {
        const QkvRopeLaunch &r = *rope;
        if (!(r.head_dim == 64 || r.head_dim == 128))
            return fa_fail(FA_ERR_OPERATION_NOT_SUPPORTED, "FusedQkv with the KvPrepFused write stage supports head_dim 64 or 128, got %u", r.head_dim);
        if (l.n_dim != r.n_heads * r.head_dim || l.n_kv != r.n_kv_heads * r.head_dim)
            return fa_fail(FA_ERR_INVALID_SHAPE, "Invalid shape: n_dim %u / n_kv %u are not n_heads %u / n_kv_heads %u x head_dim %u", l.n_dim,
                           l.n_kv, r.n_heads, r.n_kv_heads, r.head_dim);
        if (l.residual) return fa_fail(FA_ERR_OPERATION_NOT_SUPPORTED, "the KvPrepFused write stage takes no residual");
        if (r.table_rows == 0) return fa_fail(FA_ERR_INVALID_SHAPE, "Invalid shape: empty RoPE tables");
        a.out[0] = r.q_rot, a.out[1] = r.k_cache, a.out[2] = r.v_cache;
        RopeDev &d = a.r;
        d.cos_t = r.cos_t, d.sin_t = r.sin_t, d.block_table = r.block_table;
        d.on = 1, d.head_dim = r.head_dim, d.n_kv_heads = r.n_kv_heads, d.position_offset = r.position_offset;
        d.max_seq_len = r.max_seq_len, d.block_size = r.block_size ? r.block_size : 1, d.capacity = r.capacity;
        d.table_rows = r.table_rows, d.normal = r.rope_normal ? 1u : 0u, d.apply = r.apply_rope ? 1u : 0u;
        a.block_shift = (d.block_size & (d.block_size - 1)) == 0 ? (uint32_t)__builtin_ctz(d.block_size) : 32u;
    }
    const fa_panel::Plan p = fa_panel::panel_plan(panel_shape(l, rope != nullptr), ctx->n_cus > 0 ? (uint32_t)ctx->n_cus : 256u);
    a.rows_per_wg = p.rows_per_wg, a.n_pass = p.n_pass, a.beside = p.beside(), a.inv_beside = a.beside ? fa_inverse(a.beside) : 0;
    a.scale_pairs = l.k_dim / 32 % 2 == 0 ? 1u : 0u;
    for (int i = 0; i < 3; ++i)
        if (reinterpret_cast<uintptr_t>(l.scales[i]) % 4 != 0) a.scale_pairs = 0;
    FaLaunchScope scope(ctx, rope ? "fused_qkv_rows32_rope_kernel" : l.n_kv ? "fused_qkv_rows32_kernel" : "matmul_rows32_kernel", true);
    const bool sums = l.m < FA_GEMM_MIN_M_DEFAULT;  // (of interest to block-quantised weights only: the arithmetic, see fa_panel.h)
    if (l.weight_bits == 16) FA_TRY(fa_panel::launch<16>(scope, rope != nullptr, sums, p, a));
    else if (l.weight_bits == 8) FA_TRY(fa_panel::launch<8>(scope, rope != nullptr, sums, p, a));
    else FA_TRY(fa_panel::launch<4>(scope, rope != nullptr, sums, p, a));
    return scope.finish();
}

// FusedQkv + KvPrepFused of a chunk that the panel kernel takes, as one launch.
fa_status fa_launch_fused_qkv_rows32_rope(fa_ctx *ctx, const FusedQkvLaunch &l, const QkvRopeLaunch &r) {
    if (!fa_qkv_rows32_takes(ctx, l)) return fa_fail(FA_ERR_INVALID_OPERATION, "fa_launch_fused_qkv_rows32_rope: not a launch of the panel kernel");
    return launch_panel(ctx, l, &r);
}

fa_status fa_launch_fused_qkv(fa_ctx *ctx, const FusedQkvLaunch &l, bool weight_stream_only) {
    if (l.m == 1 && !(ctx->gemm_min_m == 1 && !weight_stream_only)) {
        bool taken = false;
        FA_TRY(fa_launch_gemv_row(ctx, l, &taken));
        if (taken) return FA_OK;
    }
    QkvDev a;
    for (int i = 0; i < 3; ++i) a.w[i] = l.w[i], a.bias[i] = l.bias[i], a.out[i] = l.out[i];
    a.rows[0] = l.n_dim, a.rows[1] = l.n_kv, a.rows[2] = l.n_kv;
    a.x = l.x, a.gamma = l.gamma, a.k_dim = l.k_dim, a.m = l.m, a.eps = l.eps, a.canonical = l.canonical ? 1u : 0u;
    a.residual = l.residual, a.alpha = l.alpha, a.beta = l.beta;
    for (int i = 0; i < 3; ++i) a.scales[i] = l.scales[i];
    a.rcp_nkb = l.k_dim / 32 > 1 ? (uint32_t)((1ull << 32) / (l.k_dim / 32)) + 1u : 0u;
    const bool q8 = l.scales[0] != nullptr;
    const bool q4 = l.weight_bits == 4;
    // More than a few input rows: no longer a weight stream but a GEMM (fa_gemm.hip). Measured on 5120 x 3072 with a
    // gamma, this kernel against the GEMM (norm kernel, split-K GEMM, finish kernel): m = 4: 10.4 / 16.7 us, m = 10:
    // 13.8 / 16.9, m = 12 (from where only one workgroup's input rows fit a CU's LDS): 18.8 / 17.0, m = 16: 19.7 / 17.5,
    // m = 24 (two passes): 35.1 / 18.2.
    static_assert(fa_panel::BLOCK_SUMS_BELOW == FA_GEMM_MIN_M_DEFAULT, "the panel kernel follows the weight stream's arithmetic below the GEMM's");
    constexpr uint32_t GEMM_MIN_M_DEFAULT = FA_GEMM_MIN_M_DEFAULT;
    auto aligned16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    const bool gemm_ok = l.k_dim % (q8 ? 32 : 8) == 0 && aligned16(l.x) && aligned16(l.w[0]) && aligned16(l.w[1]) &&
                         aligned16(l.w[2]) && aligned16(l.gamma);
    const uint32_t total_rows = l.n_dim + 2 * l.n_kv;
    const uint32_t n_cus = ctx->n_cus > 0 ? (uint32_t)ctx->n_cus : 256u;
    // A chunk of a few dozen input rows (the reference's default prefill chunk is 32) is still a weight stream: one launch where
    // the GEMM route takes two or three.
    if (fa_qkv_rows32_takes(ctx, l)) return launch_panel(ctx, l, nullptr);
    if (!weight_stream_only && gemm_ok && l.m >= (ctx->gemm_min_m ? ctx->gemm_min_m : GEMM_MIN_M_DEFAULT)) return fa_launch_fused_qkv_gemm(ctx, l);
    // Workgroups: a multiple of the CU count, enough of them that a workgroup's rows fit one 16-row tile where the
    // matrix allows (5120 rows, 256 CUs: 512 workgroups of 10 rows, two resident per CU - every CU requests the same
    // bytes, and all of a wave's blocks are in flight at once); at most 64 rows (4 tiles) per workgroup. Measured on
    // 5120 x 3072: 10 rows 9.35 us, 16 rows (320 workgroups) 9.18, 20 rows (one workgroup per CU, two tiles) 10.8,
    // 8 rows (640 workgroups, a third of them waiting for a slot) 13.3.
    uint32_t n_wg = n_cus * ceil_div_u32(ceil_div_u32(total_rows, 16), n_cus);
    uint32_t rows_per_wg = ceil_div_u32(total_rows, n_wg);
    if (rows_per_wg > 64) rows_per_wg = 64;
    a.rows_per_wg = rows_per_wg;
    a.x_stride = l.k_dim * 2 + 64;  // 64 bytes of padding: the 64 lanes of an operand read fall into different banks
    const uint32_t lds_budget = 128u * 1024u;
    uint32_t cols = lds_budget / a.x_stride;
    if (cols == 0) return fa_fail(FA_ERR_OPERATION_NOT_SUPPORTED, "FusedQkv: k_dim %u is too large for one input row in LDS", l.k_dim);
    if (cols > 16) cols = 16;
    if (cols > l.m) cols = l.m;
    a.cols_per_pass = cols;
    const uint32_t tiles_per_wg = ceil_div_u32(rows_per_wg, 16);
    const size_t lds = (size_t)cols * a.x_stride + (size_t)QKV_NW * 16 * 17 * sizeof(float) +
                       (q8 ? (size_t)tiles_per_wg * 16 * (l.k_dim / 32) * 2 : 0);
    static std::atomic<bool> lds_allowed_on[64];  // per device (contexts of several threads may get here together: the calls are idempotent)
    std::atomic<bool> &lds_allowed = lds_allowed_on[ctx->device & 63];
    if (!lds_allowed.load(std::memory_order_acquire)) {
        FA_HIP(hipFuncSetAttribute((const void *)fused_qkv_kernel<16>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)(lds_budget + 16 * 1024)));
        FA_HIP(hipFuncSetAttribute((const void *)fused_qkv_kernel<8>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)(lds_budget + 16 * 1024)));
        FA_HIP(hipFuncSetAttribute((const void *)fused_qkv_kernel<4>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)(lds_budget + 16 * 1024)));
        lds_allowed.store(true, std::memory_order_release);
    }
    const dim3 grid(ceil_div_u32(total_rows, rows_per_wg), ceil_div_u32(l.m, cols));
    if (grid.y > 65535u) return fa_fail(FA_ERR_INVALID_SHAPE, "Invalid shape: FusedQkv m %u needs %u passes", l.m, grid.y);
    FaLaunchScope scope(ctx, l.n_kv ? "fused_qkv_kernel" : "matmul_gemv_kernel", true);
    if (lds > lds_budget + 16 * 1024) return fa_fail(FA_ERR_OPERATION_NOT_SUPPORTED, "FusedQkv: k_dim %u needs %zu bytes of LDS", l.k_dim, lds);
    if (q4) scope.launch(fused_qkv_kernel<4>, grid, dim3(QKV_NT), lds, a);
    else if (q8) scope.launch(fused_qkv_kernel<8>, grid, dim3(QKV_NT), lds, a);
    else scope.launch(fused_qkv_kernel<16>, grid, dim3(QKV_NT), lds, a);
    return scope.finish();
}
