// FusedQkv and MatMul for many input rows (a prefill chunk): a tiled f16 GEMM on the matrix cores; F16, Q8_0 or Q4_0 weights.
// Reference: the same ops as fa_qkv.hip - src/metals/gemv/qkv_step.rs:14-120 (FusedQkv), src/metals/matmul.rs:190-239
// (MatMul; its large-m form is a GEMM, src/metals/mma) - with the write stage of src/metals/gemv/stages.rs:200-224.
//
// With more than a few input rows the step is no longer a weight stream: out[m, n] = x[m, :] . W[n, :] is
// 2 * m * n * k flops on m * k + n * k operands, so it runs as a GEMM. Almost every launch goes to the tile kernels of fa_tile.h
// (choose_tile below); this file holds the normalisation in front of them and the kernel that takes every other shape, and few tiles
// over many features:
//   * a workgroup (4 waves) owns a 128 (weight rows) x 128 (input rows) output tile; a wave owns 64 x 64 of it as
//     2 x 2 v_mfma_f32_32x32x16_f16 tiles (64 accumulator registers);
//   * both operands move through registers and LDS in steps of 64 features, two stages, one barrier per step;
//   * LDS layouts are chosen so that writes (served 8 lanes at a time) and operand reads (16 lanes at a
//     time) are free of bank conflicts; the blocked ("canonical") weight layout is one contiguous 8 KiB per (tile, 32
//     features);
//   * the rows of W_q, W_k, W_v are tiled per matrix (a tile never straddles two); the workgroups of one XCD take
//     consecutive tiles of the weight rows over all input rows, so a weight tile is fetched into one L2 only;
//   * epilogue: accumulators to LDS as f32 [input row][weight row], then alpha * sum + bias + beta * residual, one
//     rounding to f16 (as the GEMV path), 16-byte token-major stores - or, with a RoPE write stage, the KvPrepFused
//     arithmetic on those f16 values and stores to q_rot and the cache rows (rope_store_piece).
// RMSNorm: a small kernel in front writes the normalised input, rounded to f16 as qkv_project.metal:66-67 does, into
// the context's workspace; the GEMM reads that. Launches with few output tiles divide a tile's feature steps over
// several workgroups (f32 partial tiles in the workspace, added in split order by gemm_finish_kernel).
#include "fa_gemm.h"
#include "fa_norm.h"
#include "fa_tile.h"
#include <algorithm>
#include <atomic>
#include <type_traits>

namespace {

constexpr int GM_NT = 256;
constexpr int GM_TN = 128, GM_TM = 128, GM_BK = 64;
constexpr int GM_PIECES = GM_BK / 8;                   // 16-byte pieces of a row per step
// Piece stride in LDS, in bytes. An LDS write of 16 bytes per lane is served 8 lanes (128 bytes) at a time, and the 8
// must fall into different 16-byte bank groups: with the stride an odd number of pieces when 8 consecutive lanes hold
// the 8 pieces of one row, and 2 (mod 8) pieces when they hold 4 pieces of 2 rows. (Measured: with 130 and 132
// pieces a third of the LDS cycles were bank conflicts. Giving consecutive lanes consecutive rows instead also
// removes them, but such a request touches 64 cache lines instead of 8 and the loads get slower by more.)
constexpr int GM_STRIDE_ROWMAJOR = GM_TN * 16 + 16;    // a wave's 64 loads are 8 rows x 8 pieces
constexpr int GM_STRIDE_CANONICAL = GM_TN * 16 + 32;   // ... 16 rows x 4 pieces
constexpr int GM_OPERAND_BYTES = GM_PIECES * GM_STRIDE_CANONICAL;  // the larger of the two
constexpr int GM_STAGE_BYTES = 2 * GM_OPERAND_BYTES;
constexpr int GM_T_STRIDE = GM_TN * 4 + 16;             // epilogue tile: bytes per input row
constexpr int GM_LDS_BYTES = 2 * GM_STAGE_BYTES > GM_TM * GM_T_STRIDE ? 2 * GM_STAGE_BYTES : GM_TM * GM_T_STRIDE;
constexpr int GM_LOADS = GM_TN * GM_PIECES / GM_NT;     // 16-byte pieces per thread, operand and step (4)

using namespace fa_gemm;

// inv_rms of each input row, then (x * inv_rms) * gamma in f32, rounded to f16 (rmsnorm.metal:17-96). A wave takes a row: all of it
// is requested at once, kept in registers (P pieces of 16 bytes per lane) and read once, and no wave waits for another.
constexpr int NORM_ROWS = 4;  // rows (waves) per workgroup
template <int P>
__global__ void __launch_bounds__(NORM_ROWS * 64) rmsnorm_rows_kernel(const __half *x, const __half *gamma, __half *y, uint32_t m, uint32_t K,
                                                                      float inv_k, float eps) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t row = blockIdx.x * NORM_ROWS + wave;
    if (row >= m) return;
    const __half *xr = x + (size_t)row * K;
    __half *yr = y + (size_t)row * K;
    h8_t v[P], g[P];
#pragma unroll
    for (int i = 0; i < P; ++i) v[i] = *reinterpret_cast<const h8_t *>(xr + min((uint32_t)(lane + 64 * i) * 8, K - 8));
#pragma unroll
    for (int i = 0; i < P; ++i) g[i] = *reinterpret_cast<const h8_t *>(gamma + min((uint32_t)(lane + 64 * i) * 8, K - 8));
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const h8_t z = {0, 0, 0, 0, 0, 0, 0, 0}, u = (uint32_t)(lane + 64 * i) * 8 < K ? v[i] : z;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += (float)u[e] * (float)u[e];
    }
    const float inv_rms = fa_norm::inv_rms(fa_norm::wave_sum(ss), inv_k, eps);
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const h8_t o = fa_norm::scale8(v[i], inv_rms, g[i]);
        if ((uint32_t)(lane + 64 * i) * 8 < K) *reinterpret_cast<h8_t *>(yr + (uint32_t)(lane + 64 * i) * 8) = o;
    }
}
// The same for rows of more than 4096 features: a workgroup per row, which is read twice.
__global__ void __launch_bounds__(256) rmsnorm_long_rows_kernel(const __half *x, const __half *gamma, __half *y, uint32_t K, float inv_k,
                                                                float eps) {
    __shared__ float red[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const __half *xr = x + (size_t)blockIdx.x * K;
    __half *yr = y + (size_t)blockIdx.x * K;
    float ss = 0.0f;
    for (uint32_t k8 = tid; k8 < K / 8; k8 += 256) {
        const h8_t v = *reinterpret_cast<const h8_t *>(xr + k8 * 8);
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += (float)v[i] * (float)v[i];
    }
    ss = fa_norm::wave_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    const float inv_rms = fa_norm::inv_rms(((red[0] + red[1]) + red[2]) + red[3], inv_k, eps);
    for (uint32_t k8 = tid; k8 < K / 8; k8 += 256)
        *reinterpret_cast<h8_t *>(yr + k8 * 8) =
            fa_norm::scale8(*reinterpret_cast<const h8_t *>(xr + k8 * 8), inv_rms, *reinterpret_cast<const h8_t *>(gamma + k8 * 8));
}

// The end of an output tile, shared by the GEMM kernels: accumulators -> LDS (f32, [input row][weight row]) -> either
// the write stage and token-major f16 stores, or (features divided) the f32 partial tile.
__device__ __forceinline__ void gemm_epilogue(const GemmDev &a, unsigned char *smem, const f16v_t (&acc)[2][2], int tid,
                                              int lane, int wn, int wm, int mat, uint32_t N, uint32_t n0, uint32_t m0,
                                              uint32_t split) {
    const __half *bias = mat == 0 ? a.bias[0] : mat == 1 ? a.bias[1] : a.bias[2];
    __half *out = mat == 0 ? a.out[0] : mat == 1 ? a.out[1] : a.out[2];
    const uint32_t col0 = (mat >= 1 ? a.rows[0] : 0u) + (mat == 2 ? a.rows[1] : 0u) + n0;
    // Accumulators -> LDS as f32 [input row][weight row]. Register r of lane l of a 32 x 32 tile is weight row
    // 8 (r / 4) + 4 (l / 32) + r % 4 and input row l % 32: four consecutive weight rows per 16-byte write.
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const uint32_t nrow = wn * 64 + i * 32 + g * 8 + (lane >> 5) * 4;
                const uint32_t trow = wm * 64 + j * 32 + (lane & 31);
                const f4v_t q = {acc[i][j][g * 4 + 0], acc[i][j][g * 4 + 1], acc[i][j][g * 4 + 2], acc[i][j][g * 4 + 3]};
                *reinterpret_cast<f4v_t *>(smem + trow * GM_T_STRIDE + nrow * 4) = q;
            }
        }
    __syncthreads();

    if (a.k_splits > 1) {  // partial sums only; the write stage runs in gemm_finish_kernel
        for (uint32_t q = tid; q < (uint32_t)GM_TM * GM_TN / 4; q += GM_NT) {
            const uint32_t t = q / (GM_TN / 4), n4 = q % (GM_TN / 4);
            const uint32_t gm = m0 + t, gn = n0 + n4 * 4;
            if (gm >= a.m || gn >= N) continue;
            const f4v_t s = *reinterpret_cast<const f4v_t *>(smem + t * GM_T_STRIDE + n4 * 16);
            float *dst = a.partial + ((size_t)split * a.m + gm) * a.n_total + col0 + n4 * 4;
            if (a.vec_store) {
                *reinterpret_cast<f4v_t *>(dst) = s;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (gn + e < N) dst[e] = s[e];
            }
        }
        return;
    }
    for (uint32_t q = tid; q < (uint32_t)GM_TM * GM_TN / 8; q += GM_NT) {
        const uint32_t t = q / (GM_TN / 8), n8 = q % (GM_TN / 8);
        const uint32_t gm = m0 + t, gn = n0 + n8 * 8;
        if (gm >= a.m || gn >= N) continue;
        const f4v_t s0 = *reinterpret_cast<const f4v_t *>(smem + t * GM_T_STRIDE + n8 * 32);
        const f4v_t s1 = *reinterpret_cast<const f4v_t *>(smem + t * GM_T_STRIDE + n8 * 32 + 16);
        const size_t o = (size_t)gm * N + gn;
        if (a.vec_store) {  // N % 8 == 0 and 16-byte aligned tensors: whole pieces
            const h8_t z = {0, 0, 0, 0, 0, 0, 0, 0};
            const h8_t bv = bias ? *reinterpret_cast<const h8_t *>(bias + gn) : z;
            const h8_t rv = a.residual ? *reinterpret_cast<const h8_t *>(a.residual + o) : z;
            h8_t y;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float v = (e < 4 ? s0[e & 3] : s1[e & 3]) * a.alpha;
                if (bias) v += (float)bv[e];
                if (a.residual) v += a.beta * (float)rv[e];
                y[e] = (_Float16)v;
            }
            if (a.rope.on) {
                // the mate piece of a NeoX pair lies half a head away in the same LDS row (a tile holds whole heads)
                h8_t mate = z;
                if (!a.rope.normal && a.rope.apply && mat != 2) {
                    const uint32_t hp = a.rope.head_dim >> 4;  // pieces in half a head
                    const uint32_t m8 = ((n8 * 8) & (a.rope.head_dim - 1)) < (a.rope.head_dim >> 1) ? n8 + hp : n8 - hp;
                    const f4v_t t0 = *reinterpret_cast<const f4v_t *>(smem + t * GM_T_STRIDE + m8 * 32);
                    const f4v_t t1 = *reinterpret_cast<const f4v_t *>(smem + t * GM_T_STRIDE + m8 * 32 + 16);
                    const h8_t bm = bias ? *reinterpret_cast<const h8_t *>(bias + n0 + m8 * 8) : z;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        float v = (e < 4 ? t0[e & 3] : t1[e & 3]) * a.alpha;
                        if (bias) v += (float)bm[e];
                        mate[e] = (_Float16)v;
                    }
                }
                rope_store_piece(a, mat, gm, gn, y, mate);
            } else {
                *reinterpret_cast<h8_t *>(out + o) = y;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (gn + e >= N) break;
                float v = (e < 4 ? s0[e & 3] : s1[e & 3]) * a.alpha;
                if (bias) v += __half2float(bias[gn + e]);
                if (a.residual) v += a.beta * __half2float(a.residual[o + e]);
                out[o + e] = __float2half(v);
            }
        }
    }
}

// Block-quantised weights become f16 on their way into LDS as the reference's GEMM tile loader makes them
// (src/metals/mma/tile_loader.metal:100-120: (half)(weight * (float)scale); the CPU reference of its tests dequantises
// the same way, tests/gemm_v2_parity.rs:295-350): the integer is converted exactly, then multiplied by its block's scale
// with one f16 rounding. From there on the GEMM is the F16 one. (The weight-stream kernel keeps the GEMV policies'
// arithmetic instead - block sums in f32 times the scale; an earlier form of this kernel did that too, with 64 scaled
// adds per block and wave beside 8 matrix instructions, and was bound by them: 152 us against 121 for F16 on 2048 x
// 5120 x 3072.)
// WB: bits per weight - 16 (f16), 8 (Q8_0) or 4 (Q4_0: 16 bytes are the 32 features of a block = four f16 pieces).
template <bool CANON, int WB>
__global__ void __launch_bounds__(GM_NT, 2) qkv_gemm_kernel(GemmDev a) {
    constexpr bool Q8 = WB != 16;  // block-quantised: integer weights with one f16 scale per 32 of a row
    constexpr bool Q4 = WB == 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    constexpr int W_STRIDE = CANON ? GM_STRIDE_CANONICAL : GM_STRIDE_ROWMAJOR;
    constexpr int X_STRIDE = GM_STRIDE_ROWMAJOR;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t K = a.k_dim;

    // Tile of this workgroup. Workgroup ids go round the 8 XCDs; the ids of one XCD are given consecutive tiles.
    const uint32_t total = a.n_tiles * a.m_tiles * a.k_splits;
    uint32_t v = blockIdx.x;
    if (total % 8 == 0) v = (blockIdx.x % 8) * (total / 8) + blockIdx.x / 8;
    const uint32_t split = v % a.k_splits;
    v /= a.k_splits;
    uint32_t nt = v / a.m_tiles;
    const uint32_t mt = v - nt * a.m_tiles;
    int mat = 0;
    if (nt >= a.tiles[0]) {
        nt -= a.tiles[0], mat = 1;
        if (nt >= a.tiles[1]) nt -= a.tiles[1], mat = 2;
    }
    const uint32_t N = mat == 0 ? a.rows[0] : a.rows[1];
    const unsigned char *W = reinterpret_cast<const unsigned char *>(mat == 0 ? a.w[0] : mat == 1 ? a.w[1] : a.w[2]);
    const uint32_t n0 = nt * GM_TN, m0 = mt * GM_TM;

    // Global pieces of this thread: GM_LOADS 16-byte pieces per operand and step (Q8 weights: half as many).
    //   weights, canonical: piece p = tid + 256 i of a step = (32-feature block p / 512, row (p % 512) / 4, piece p % 4)
    //   weights, row-major and input: piece p = (row p / 8, piece p % 8)
    //   Q8 weights: 16 bytes are 16 features = two f16 pieces; canonical (block i, row tid / 2, half tid % 2),
    //   row-major (row p / 4, quarter p % 4)
    //   Q4 weights: 16 bytes are the 32 features of one block = four f16 pieces; canonical (block tid / 128, row
    //   tid % 128), row-major (row tid / 2, block tid % 2)
    constexpr int W_LOADS = Q4 ? 1 : Q8 ? GM_LOADS / 2 : GM_LOADS;
    const unsigned char *wp[W_LOADS];
    const unsigned char *xp[GM_LOADS];
    uint32_t w_lds[W_LOADS], x_lds[GM_LOADS];
    bool w_ok[W_LOADS], x_ok[GM_LOADS];
    uint32_t w_kpiece[W_LOADS];  // first feature of the piece within the step, for the tail guard
    uint32_t w_row[W_LOADS];
    uint32_t x_kpiece[GM_LOADS];
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) {
        const uint32_t p = tid + GM_NT * i;
        uint32_t row, piece;
        if constexpr (Q4) {
            if (CANON) {
                row = tid % GM_TN, piece = (tid / GM_TN) * 4;
                wp[i] = W + ((size_t)(n0 + row) * 32 + (size_t)(tid / GM_TN) * N * 32) / 2;
            } else {
                row = tid / 2, piece = (tid % 2) * 4;
                wp[i] = W + ((size_t)(n0 + row) * K + (tid % 2) * 32) / 2;
            }
        } else if constexpr (Q8) {
            if (CANON) {
                row = tid / 2, piece = i * 4 + (tid % 2) * 2;
                wp[i] = W + (size_t)(n0 + row) * 32 + (size_t)i * N * 32 + (tid % 2) * 16;
            } else {
                row = p / 4, piece = (p % 4) * 2;
                wp[i] = W + (size_t)(n0 + row) * K + (p % 4) * 16;
            }
        } else if (CANON) {
            const uint32_t blk = p / 512, within = p % 512;
            row = within / 4, piece = blk * 4 + within % 4;
            wp[i] = W + ((size_t)(n0 + row) * 32 + (size_t)blk * N * 32 + (within % 4) * 8) * 2;
        } else {
            row = p / 8, piece = p % 8;
            wp[i] = W + ((size_t)(n0 + row) * K + piece * 8) * 2;
        }
        w_ok[i] = n0 + row < N;
        w_lds[i] = piece * W_STRIDE + row * 16;
        w_kpiece[i] = piece * 8;
        w_row[i] = row;
    }
#pragma unroll
    for (int i = 0; i < GM_LOADS; ++i) {
        const uint32_t p = tid + GM_NT * i;
        const uint32_t xrow = p / 8, xpiece = p % 8;
        xp[i] = reinterpret_cast<const unsigned char *>(a.x) + ((size_t)(m0 + xrow) * K + xpiece * 8) * 2;
        x_ok[i] = m0 + xrow < a.m;
        x_lds[i] = xpiece * X_STRIDE + xrow * 16;
        x_kpiece[i] = xpiece * 8;
    }
    const size_t w_step = (CANON ? (size_t)2 * N * 32 : (size_t)GM_BK) * WB / 8;  // bytes between steps
    const size_t x_step = (size_t)GM_BK * 2;
    // Block-quantised weights: each 16-byte request lies within one 32-feature block of one row; its scale
    // (scales[row][k_dim / 32]) is requested with it and folded into the f16 weights on their way into LDS.
    const uint32_t nkb = K / 32;
    const __half *w_scale[W_LOADS];
    if constexpr (Q8) {
        const __half *sp = mat == 0 ? a.scales[0] : mat == 1 ? a.scales[1] : a.scales[2];
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i) w_scale[i] = sp + (size_t)(n0 + w_row[i]) * nkb + w_kpiece[i] / 32;
    }

    typedef typename std::conditional<Q8, u4v_t, h8_t>::type wreg_t;
    wreg_t wr[W_LOADS];
    h8_t xr[GM_LOADS];
    _Float16 wsc[W_LOADS];
    auto fetch = [&](uint32_t ks) {
        const uint32_t k0 = ks * GM_BK;
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i) {
            wreg_t z;
            if constexpr (Q8) z = u4v_t{0u, 0u, 0u, 0u};
            else z = h8_t{0, 0, 0, 0, 0, 0, 0, 0};
            const bool ok = w_ok[i] && k0 + w_kpiece[i] < K;
            wr[i] = ok ? *reinterpret_cast<const wreg_t *>(wp[i] + ks * w_step) : z;
            if constexpr (Q8) wsc[i] = ok ? *reinterpret_cast<const _Float16 *>(w_scale[i] + ks * 2) : (_Float16)0.0f;
        }
#pragma unroll
        for (int i = 0; i < GM_LOADS; ++i) {
            const h8_t z = {0, 0, 0, 0, 0, 0, 0, 0};
            xr[i] = (x_ok[i] && k0 + x_kpiece[i] < K) ? *reinterpret_cast<const h8_t *>(xp[i] + ks * x_step) : z;
        }
    };
    auto stash = [&](int stage) {
        unsigned char *base = smem + stage * GM_STAGE_BYTES;
#pragma unroll
        for (int i = 0; i < W_LOADS; ++i) {
            if constexpr (Q4) {
                const h8_t sc = {wsc[i], wsc[i], wsc[i], wsc[i], wsc[i], wsc[i], wsc[i], wsc[i]};
#pragma unroll
                for (int q = 0; q < 4; ++q) *reinterpret_cast<h8_t *>(base + w_lds[i] + q * W_STRIDE) = fa_quant::q4_to_f16(wr[i][q]) * sc;
            } else if constexpr (Q8) {
                const h8_t sc = {wsc[i], wsc[i], wsc[i], wsc[i], wsc[i], wsc[i], wsc[i], wsc[i]};
                *reinterpret_cast<h8_t *>(base + w_lds[i]) = fa_quant::q8_to_f16(wr[i][0], wr[i][1]) * sc;
                *reinterpret_cast<h8_t *>(base + w_lds[i] + W_STRIDE) = fa_quant::q8_to_f16(wr[i][2], wr[i][3]) * sc;
            } else {
                *reinterpret_cast<h8_t *>(base + w_lds[i]) = wr[i];
            }
        }
#pragma unroll
        for (int i = 0; i < GM_LOADS; ++i) *reinterpret_cast<h8_t *>(base + GM_OPERAND_BYTES + x_lds[i]) = xr[i];
    };

    // Wave (wn, wm) owns weight rows 64 wn .. +63 and input rows 64 wm .. +63 of the tile.
    const int wn = wave & 1, wm = wave >> 1;
    const uint32_t a_off = (lane >> 5) * W_STRIDE + (wn * 64 + (lane & 31)) * 16;
    const uint32_t b_off = (lane >> 5) * X_STRIDE + (wm * 64 + (lane & 31)) * 16;
    f16v_t acc[2][2], sums[2][2];  // (F16: of the last steps, and of all before, where the tile kernels add them up)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = sums[i][j][r] = 0.0f;

    const uint32_t all_steps = (K + GM_BK - 1) / GM_BK;
    const uint32_t ks_begin = split * a.steps_per_split;
    const uint32_t n_steps = min(all_steps, ks_begin + a.steps_per_split);  // end of this workgroup's range
    fetch(ks_begin);
    stash(ks_begin & 1);
    __syncthreads();
    for (uint32_t ks = ks_begin; ks < n_steps; ++ks) {
        const bool more = ks + 1 < n_steps;
        if (more) fetch(ks + 1);
        if (WB == 16 && (ks - ks_begin) % 4 == 3) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) sums[i][j] += acc[i][j], acc[i][j] = f16v_t{};
        }
        const unsigned char *wa = smem + (ks & 1) * GM_STAGE_BYTES;
        const unsigned char *xa = wa + GM_OPERAND_BYTES;
        {
#pragma unroll
            for (int kk = 0; kk < GM_BK / 16; ++kk) {
                h8_t fa[2], fb[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    fa[i] = *reinterpret_cast<const h8_t *>(wa + a_off + kk * 2 * W_STRIDE + i * 32 * 16);
                    fb[i] = *reinterpret_cast<const h8_t *>(xa + b_off + kk * 2 * X_STRIDE + i * 32 * 16);
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i], fb[j], acc[i][j], 0, 0, 0);
            }
        }
        if (more) stash((ks + 1) & 1);
        __syncthreads();
    }

    if constexpr (WB == 16) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = sums[i][j] + acc[i][j];
    }
    gemm_epilogue(a, smem, acc, tid, lane, wn, wm, mat, N, n0, m0, split);
}

// Adds the partial tiles in split order and applies the write stage: one thread per 8 output columns.
__global__ void __launch_bounds__(256) gemm_finish_kernel(GemmDev a) {
    const uint32_t groups = (a.n_total + 7) / 8;
    const uint32_t id = blockIdx.x * 256 + threadIdx.x;
    if (id >= a.m * groups) return;
    const uint32_t gm = id / groups, col = (id - gm * groups) * 8;
    int mat = 0;
    uint32_t gn = col;
    if (gn >= a.rows[0]) {
        gn -= a.rows[0], mat = 1;
        if (gn >= a.rows[1]) gn -= a.rows[1], mat = 2;
    }
    const uint32_t N = mat == 0 ? a.rows[0] : a.rows[1];
    const __half *bias = mat == 0 ? a.bias[0] : mat == 1 ? a.bias[1] : a.bias[2];
    __half *out = mat == 0 ? a.out[0] : mat == 1 ? a.out[1] : a.out[2];
    const size_t o = (size_t)gm * N + gn;
    if (a.vec_store) {
        const size_t split_stride = (size_t)a.m * a.n_total;
        const h8_t z = {0, 0, 0, 0, 0, 0, 0, 0};
        // the write stage's value of the 8 columns from column c of the concatenated list (column g of the matrix)
        auto piece = [&](uint32_t c, uint32_t g) -> h8_t {
            f4v_t s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = s0;
            const float *src = a.partial + (size_t)gm * a.n_total + c;
            uint32_t sp = 0;
            for (; sp + 4 <= a.k_splits; sp += 4) {  // four splits' loads in flight, added in split order
                f4v_t u[4], w[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    u[q] = *reinterpret_cast<const f4v_t *>(src + (sp + q) * split_stride);
                    w[q] = *reinterpret_cast<const f4v_t *>(src + (sp + q) * split_stride + 4);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) s0 += u[q], s1 += w[q];
            }
            for (; sp < a.k_splits; ++sp) {
                s0 += *reinterpret_cast<const f4v_t *>(src + sp * split_stride);
                s1 += *reinterpret_cast<const f4v_t *>(src + sp * split_stride + 4);
            }
            const h8_t bv = bias ? *reinterpret_cast<const h8_t *>(bias + g) : z;
            const h8_t rv = a.residual ? *reinterpret_cast<const h8_t *>(a.residual + (size_t)gm * N + g) : z;
            h8_t y;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float t = (e < 4 ? s0[e & 3] : s1[e & 3]) * a.alpha;
                if (bias) t += (float)bv[e];
                if (a.residual) t += a.beta * (float)rv[e];
                y[e] = (_Float16)t;
            }
            return y;
        };
        const h8_t y = piece(col, gn);
        if (a.rope.on) {
            h8_t mate = z;
            if (!a.rope.normal && a.rope.apply && mat != 2) {  // NeoX: the piece half a head away
                const uint32_t half = a.rope.head_dim >> 1;
                const bool first = (gn & (a.rope.head_dim - 1)) < half;
                mate = first ? piece(col + half, gn + half) : piece(col - half, gn - half);
            }
            rope_store_piece(a, mat, gm, gn, y, mate);
        } else {
            *reinterpret_cast<h8_t *>(out + o) = y;
        }
    } else {
        // a group of 8 columns of the concatenated list may straddle two matrices: element by element
        for (uint32_t e = 0; e < 8 && col + e < a.n_total; ++e) {
            int me = 0;
            uint32_t ge = col + e;
            if (ge >= a.rows[0]) {
                ge -= a.rows[0], me = 1;
                if (ge >= a.rows[1]) ge -= a.rows[1], me = 2;
            }
            const uint32_t Ne = me == 0 ? a.rows[0] : a.rows[1];
            const __half *be = me == 0 ? a.bias[0] : me == 1 ? a.bias[1] : a.bias[2];
            __half *oe = me == 0 ? a.out[0] : me == 1 ? a.out[1] : a.out[2];
            float s = 0.0f;
            for (uint32_t sp = 0; sp < a.k_splits; ++sp) s += a.partial[((size_t)sp * a.m + gm) * a.n_total + col + e];
            float t = s * a.alpha;
            if (be) t += __half2float(be[ge]);
            if (a.residual) t += a.beta * __half2float(a.residual[(size_t)gm * Ne + ge]);
            oe[(size_t)gm * Ne + ge] = __float2half(t);
        }
    }
}

}  // namespace

// The cheapest tile shape for a launch over rows[i] weight rows per matrix, and its cost: what a tile of each shape takes per step of
// 64 features with one workgroup on every CU, in units of the 64 x 64 tile's 0.21 us (from launches of 160 to 256 tiles over 3072
// features), times the rounds of workgroups that the launch has. The larger tiles read less per product, the smaller ones leave
// fewer CUs idle: 64 x 96 is for 257 to 384 tiles of 64 x 64, which are one round of it (576 rows, 3072 x 2048 F16: 18.4 us as two
// rounds or as 128 x 64, 16.0 as 64 x 96; 500 rows 3072 x 3072, with a residual, 19.5 -> 15.9, Q8_0 17.6 -> 16.4, Q4_0 17.0 -> 15.4). Three rounds
// and more of 64 x 96, and of any small F16 tiles, take longer than their number says (2079 rows, 2048 x 2048 F16: 30.8 us in three
// rounds of 64 x 96, 27.5 in two of 128 x 128). It moves no F16 launch from the tiles that add their sums up in parts (fa_tile.h) to the
// larger ones, which do not: 1300 rows, 3072 x 3072 take 33.7 us in one round of 256 x 128 and 37.7 in four of 64 x 64, but with errors
// of 5.9 x 2^-24 of the sums' size in place of 2.2. Over 730 launches of 130 to 2200 rows the choice is on average within 0.1 % (F16), 0.5 %
// (block-quantised) of the best shape, 1.5 to 2 % without 64 x 96. `joined`: tiles may hold rows of two matrices. `variant`: a shape
// asked for by name (fa_set_gemm_variant).
static float best_tile(const FusedQkvLaunch &l, const uint32_t (&rows)[3], uint32_t n_cus, bool joined, uint32_t variant, fa_tile::TileShape &shape) {
    struct Choice {
        fa_tile::TileShape shape;
        uint32_t m, n;
        float f16, quantised;
    };
    static const Choice choices[] = {{fa_tile::TILE_64x64, 64, 64, 1.0f, 1.0f},
                                     {fa_tile::TILE_64x96, 64, 96, 1.4f, 1.4f},
                                     {fa_tile::TILE_128x64, 128, 64, 1.75f, 1.64f},
                                     {fa_tile::TILE_128x128, 128, 128, 2.6f, 2.7f},
                                     {fa_tile::TILE_256x128, 256, 128, 4.65f, 4.3f},
                                     {fa_tile::TILE_256x160, 256, 160, 6.3f, 0.0f}};
    float best = 0.0f, in_parts = 0.0f;  // (in_parts: the least by rounds alone of 64 x 64, 128 x 64 and 128 x 128, which come first)
    for (const Choice &c : choices) {
        if (c.shape == fa_tile::TILE_256x160 && !joined) continue;
        // (a block-quantised tile's scales lie in LDS over the whole of k_dim)
        if (l.weight_bits != 16 && c.shape != fa_tile::TILE_64x64 && l.k_dim > 4096) continue;
        if (variant == 2 && c.shape != fa_tile::TILE_128x128) continue;
        if (variant == 3 && c.shape != fa_tile::TILE_64x64) continue;
        uint32_t n_tiles = 0;
        for (int i = 0; i < 3; ++i) n_tiles += ceil_div_u32(rows[i], c.n);
        if (c.shape == fa_tile::TILE_256x160) n_tiles = ceil_div_u32(rows[0] + 2 * rows[1], c.n);
        const uint64_t tiles = (uint64_t)n_tiles * ceil_div_u32(l.m, c.m);
        const uint64_t rounds = (tiles + n_cus - 1) / n_cus;
        float cost = (float)rounds * (l.weight_bits == 16 ? c.f16 : c.quantised);
        if (l.weight_bits == 16 && c.m * c.n > 128 * 128 && in_parts != 0.0f && cost >= in_parts) continue;
        if (c.m * c.n <= 128 * 128 && c.shape != fa_tile::TILE_64x96) in_parts = in_parts == 0.0f ? cost : std::min(in_parts, cost);
        if (rounds >= 3 && (c.shape == fa_tile::TILE_64x96 || (l.weight_bits == 16 && c.m * c.n < 128 * 128))) cost *= 1.2f;
        if (best == 0.0f || cost < best) {
            best = cost, shape = c.shape;
            // With a workgroup or less per CU, the block-quantised form has stages for each wave, or keeps twice as many of its smaller
            // stages on their way (both measured in fa_tile.h; LDS beside the scales: up to 4096 and 8192 features).
            if (c.shape == fa_tile::TILE_64x64 && l.weight_bits != 16 && tiles <= n_cus && l.k_dim <= 8192)
                shape = l.k_dim >= 1024 && l.k_dim <= 4096 ? fa_tile::TILE_64x64_OWN : fa_tile::TILE_64x64_DEEP;
            if (c.shape == fa_tile::TILE_64x64 && l.weight_bits != 16 && variant == 0) {  // (there too; where it fills no second round)
                uint32_t narrow = 0;
                for (int i = 0; i < 3; ++i) narrow += ceil_div_u32(rows[i], 32);
                if ((uint64_t)narrow * ceil_div_u32(l.m, 64) <= n_cus) shape = fa_tile::TILE_64x32;
            }
        }
    }
    return best;
}

// How the register-staged kernel divides a launch: the feature steps of a tile over enough workgroups to give every CU a share of the
// weight stream, at least 4 steps each (512 rows of the Llama-3.2-3B projections: 42.9 -> 35.9 us with 3).
struct Division {
    uint32_t k_splits, steps_per_split;
    uint64_t n_wg;  // tiles
};
static Division divide(const FusedQkvLaunch &l, uint32_t n_cus, bool whole) {
    Division d;
    d.n_wg = (uint64_t)(ceil_div_u32(l.n_dim, GM_TN) + 2 * ceil_div_u32(l.n_kv, GM_TN)) * ceil_div_u32(l.m, GM_TM);
    const uint32_t all_steps = ceil_div_u32(l.k_dim, GM_BK);
    uint32_t splits = whole ? 1u : (uint32_t)(2 * n_cus / d.n_wg);
    if (splits > all_steps / 4) splits = all_steps / 4;
    if (splits < 1) splits = 1;
    d.steps_per_split = ceil_div_u32(all_steps, splits);
    d.k_splits = ceil_div_u32(all_steps, d.steps_per_split);
    return d;
}

// What a launch takes on the tile kernels and, divided, on the register-staged one, in us: fitted to launches of 16 to 400 rows over
// 512 to 8192 features and 512 to 10240 weight rows (on the tiles within 4 to 7 % rms, divided 8 %). The norm's launch is in both.
static float weight_mb(const FusedQkvLaunch &l) {
    return (float)l.k_dim * (float)(l.n_dim + 2 * l.n_kv) * (l.weight_bits == 16 ? 2.0f : l.weight_bits == 8 ? 1.0625f : 0.5625f) * 1e-6f;
}
static float tile_us(const FusedQkvLaunch &l, float cost) {
    const bool f16 = l.weight_bits == 16;
    const float k = (float)l.k_dim, mb = weight_mb(l);
    const float norm = l.gamma ? (f16 ? 2.3f + 3.0e-6f * (float)l.m * k : 2.0f + 2.6e-6f * (float)l.m * k) : 0.0f;
    return f16 ? 1.5f + cost * (0.137f * k / 64.0f + 1.43f) + norm + 0.076f * mb : 3.4f + cost * (0.178f * k / 64.0f + 0.1f) + norm + 0.064f * mb;
}
static float divided_us(const FusedQkvLaunch &l, const Division &d, uint32_t n_cus) {
    const float parts_mb = (float)d.k_splits * (float)l.m * (float)(l.n_dim + 2 * l.n_kv) * 4e-6f;
    const float rounds = (float)((d.n_wg * d.k_splits + 2 * n_cus - 1) / (2 * n_cus));
    return 8.0f + 0.89f * rounds * (float)d.steps_per_split + 0.35f * parts_mb + 0.094f * weight_mb(l) +
           (l.gamma ? 2.9f + 0.76e-6f * (float)l.m * (float)l.k_dim : 0.0f);
}

// What the tile kernels ask of the features, the weight rows and the scales: whole steps of 64 features, whole 16-byte stores, pairs of
// scales.
bool fa_gemm_tiles_fit(const FusedQkvLaunch &l) {
    for (int i = 0; i < 3; ++i)
        if (reinterpret_cast<uintptr_t>(l.scales[i]) % 4 != 0) return false;
    return l.k_dim % 64 == 0 && l.n_dim % 8 == 0 && l.n_kv % 8 == 0 && (l.weight_bits == 16 || l.k_dim <= 16384);
}

float fa_gemm_estimate_us(const fa_ctx *ctx, const FusedQkvLaunch &l) {
    const uint32_t n_cus = ctx->n_cus > 0 ? (uint32_t)ctx->n_cus : 256u, rows[3] = {l.n_dim, l.n_kv, l.n_kv};
    const float divided = divided_us(l, divide(l, n_cus, false), n_cus);
    fa_tile::TileShape shape;
    return fa_gemm_tiles_fit(l) ? std::min(divided, tile_us(l, best_tile(l, rows, n_cus, false, 0, shape))) : divided;
}

// Whether the tile kernels (fa_tile.h) take a launch, and with which tile: whole steps of 64 features, whole 16-byte stores, operands
// below 2 GiB (32-bit offsets).
static bool choose_tile(const fa_ctx *ctx, const FusedQkvLaunch &l, GemmDev &a, uint32_t n_cus, fa_tile::TileShape &shape) {
    const uint64_t max_rows = std::max(a.rows[0], a.rows[1]);
    if (!fa_gemm_tiles_fit(l) || !a.vec_store || (uint64_t)l.m * l.k_dim * 2 >= 0x7fffffffull || max_rows * l.k_dim * 2 >= 0x7fffffffull) return false;
    const bool joined = l.weight_bits == 16 && a.rows[0] % 32 == 0 && a.rows[1] % 32 == 0;
    const float cost = best_tile(l, a.rows, n_cus, joined, ctx->gemm_variant, shape);
    if (cost == 0.0f) return false;
    if (ctx->gemm_variant != 0) return true;
    // Few tiles over many features are one long chain of steps each: divided where that is well ahead by both estimates (us, tiles and
    // divided: 16 rows, 8192 features x 1024, Q8_0 25.6, 14.4; 32 rows, 5120 x 1024, Q4_0 18.0, 12.2; 64 rows, 4096 x 512, Q8_0 14.5,
    // 11.9 | 16 rows, 4096 x 4096, Q8_0 14.8, 15.4, F16 12.8, 15.6; 100 rows, 5120 x 1536, Q8_0 21.7, 22.8), and only into partial
    // sums that the workspace of a new context holds: a recorded graph, which cannot let it grow, takes what the tiles took.
    const Division d = divide(l, n_cus, false);
    const size_t norm_bytes = l.gamma ? (size_t)l.m * l.k_dim * sizeof(__half) + 256 : 0;
    if (norm_bytes + (size_t)d.k_splits * l.m * (l.n_dim + 2 * l.n_kv) * sizeof(float) > FA_WORKSPACE_INITIAL) return true;
    return divided_us(l, d, n_cus) >= 0.87f * tile_us(l, cost);
}

static fa_status launch_gemm(fa_ctx *ctx, const FusedQkvLaunch &l, const QkvRopeLaunch *rope) {
    if (l.k_dim % 8 != 0) return fa_fail(FA_ERR_INVALID_SHAPE, "Invalid shape: k_dim %u must be a multiple of 8", l.k_dim);
    GemmDev a;
    memset(&a, 0, sizeof(a));
    for (int i = 0; i < 3; ++i) a.w[i] = l.w[i], a.bias[i] = l.bias[i], a.out[i] = l.out[i], a.scales[i] = l.scales[i];
    if (rope) {
        const QkvRopeLaunch &r = *rope;
        // a 128-row tile of a weight matrix must hold whole heads (the NeoX mate of a column lies in the same tile)
        if (!(r.head_dim == 64 || r.head_dim == 128))
            return fa_fail(FA_ERR_OPERATION_NOT_SUPPORTED, "FusedQkv with the KvPrepFused write stage supports head_dim 64 or 128, got %u", r.head_dim);
        if (l.n_dim != r.n_heads * r.head_dim || l.n_kv != r.n_kv_heads * r.head_dim)
            return fa_fail(FA_ERR_INVALID_SHAPE, "Invalid shape: n_dim %u / n_kv %u are not n_heads %u / n_kv_heads %u x head_dim %u", l.n_dim,
                           l.n_kv, r.n_heads, r.n_kv_heads, r.head_dim);
        if (l.residual) return fa_fail(FA_ERR_OPERATION_NOT_SUPPORTED, "the KvPrepFused write stage takes no residual");
        a.out[0] = r.q_rot, a.out[1] = r.k_cache, a.out[2] = r.v_cache;
        a.rope.cos_t = r.cos_t, a.rope.sin_t = r.sin_t, a.rope.block_table = r.block_table;
        a.rope.on = 1, a.rope.head_dim = r.head_dim, a.rope.n_kv_heads = r.n_kv_heads, a.rope.position_offset = r.position_offset;
        a.rope.max_seq_len = r.max_seq_len, a.rope.block_size = r.block_size ? r.block_size : 1, a.rope.capacity = r.capacity;
        a.rope.table_rows = r.table_rows, a.rope.normal = r.rope_normal ? 1u : 0u, a.rope.apply = r.apply_rope ? 1u : 0u;
        a.page_shift = (a.rope.block_size & (a.rope.block_size - 1)) == 0 ? (uint32_t)__builtin_ctz(a.rope.block_size) : 32u;
    }
    const bool q8 = l.scales[0] != nullptr;
    a.rows[0] = l.n_dim, a.rows[1] = l.n_kv, a.rows[2] = l.n_kv;
    a.n_tiles = 0;
    for (int i = 0; i < 3; ++i) a.tiles[i] = ceil_div_u32(a.rows[i], GM_TN), a.n_tiles += a.tiles[i];
    a.k_dim = l.k_dim, a.m = l.m, a.m_tiles = ceil_div_u32(l.m, GM_TM), a.canonical = l.canonical ? 1u : 0u;
    a.residual = l.residual, a.alpha = l.alpha, a.beta = l.beta;
    a.x = l.x;
    auto aligned16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    bool vec = true;
    for (int i = 0; i < 3; ++i) {
        if (a.rows[i] == 0) continue;
        vec = vec && a.rows[i] % 8 == 0 && aligned16(a.out[i]) && (!a.bias[i] || aligned16(a.bias[i]));
    }
    vec = vec && (!a.residual || aligned16(a.residual));
    a.vec_store = vec ? 1u : 0u;
    if (rope && (!vec || !aligned16(rope->cos_t) || !aligned16(rope->sin_t)))
        return fa_fail(FA_ERR_OPERATION_NOT_SUPPORTED, "FusedQkv with the KvPrepFused write stage needs 16-byte aligned q_rot, caches, biases and tables");
    if (!aligned16(l.x) || !aligned16(l.w[0]) || (l.w[1] && !aligned16(l.w[1])) || (l.w[2] && !aligned16(l.w[2])) ||
        (l.gamma && !aligned16(l.gamma)))
        return fa_fail(FA_ERR_INVALID_SHAPE, "Invalid shape: the GEMM path needs 16-byte aligned input and weights");
    const uint64_t n_wg = (uint64_t)a.n_tiles * a.m_tiles;
    if (n_wg > 0x7fffffffull) return fa_fail(FA_ERR_INVALID_SHAPE, "Invalid shape: %llu output tiles", (unsigned long long)n_wg);
    const uint32_t n_cus = ctx->n_cus > 0 ? (uint32_t)ctx->n_cus : 256u;
    fa_tile::TileShape shape;
    const bool tiles_whole = choose_tile(ctx, l, a, n_cus, shape);
    // (What the tile kernels could take is not divided where the register-staged kernel is asked for by name: with F16 weights their
    // sums and this kernel's are the same to the bit.)
    const Division d = divide(l, n_cus, tiles_whole);
    a.steps_per_split = d.steps_per_split, a.k_splits = d.k_splits;
    a.n_total = a.rows[0] + a.rows[1] + a.rows[2];
    const size_t norm_bytes = l.gamma ? (((size_t)l.m * l.k_dim * sizeof(__half) + 255) & ~(size_t)255) : 0;
    const size_t partial_bytes = a.k_splits > 1 ? (size_t)a.k_splits * l.m * a.n_total * sizeof(float) : 0;
    if (norm_bytes + partial_bytes) FA_TRY(fa_ensure_workspace(ctx, norm_bytes + partial_bytes));
    a.partial = (float *)((char *)ctx->workspace + norm_bytes);
    if (a.k_splits > 1 && a.n_total % 8 != 0) a.vec_store = 0;  // (never with a RoPE write stage: whole heads of 64 or 128)
    if (l.gamma) {
        FaLaunchScope norm(ctx, "rmsnorm_rows_kernel", true);
        __half *y = (__half *)ctx->workspace;
        const float inv_k = 1.0f / (float)l.k_dim;
        const dim3 grid(ceil_div_u32(l.m, NORM_ROWS)), block(NORM_ROWS * 64);
        if (l.k_dim <= 1024) norm.launch(rmsnorm_rows_kernel<2>, grid, block, 0, l.x, l.gamma, y, l.m, l.k_dim, inv_k, l.eps);
        else if (l.k_dim <= 2048) norm.launch(rmsnorm_rows_kernel<4>, grid, block, 0, l.x, l.gamma, y, l.m, l.k_dim, inv_k, l.eps);
        else if (l.k_dim <= 4096) norm.launch(rmsnorm_rows_kernel<8>, grid, block, 0, l.x, l.gamma, y, l.m, l.k_dim, inv_k, l.eps);
        else norm.launch(rmsnorm_long_rows_kernel, dim3(l.m), dim3(256), 0, l.x, l.gamma, y, l.k_dim, inv_k, l.eps);
        FA_TRY(norm.finish());
        a.x = (const __half *)ctx->workspace;
    }
    static std::atomic<bool> lds_allowed_on[64];  // per device (contexts of several threads may get here together: the calls are idempotent)
    std::atomic<bool> &lds_allowed = lds_allowed_on[ctx->device & 63];
    if (!lds_allowed.load(std::memory_order_acquire)) {
        FA_HIP(hipFuncSetAttribute((const void *)qkv_gemm_kernel<false, 16>, hipFuncAttributeMaxDynamicSharedMemorySize, GM_LDS_BYTES));
        FA_HIP(hipFuncSetAttribute((const void *)qkv_gemm_kernel<true, 16>, hipFuncAttributeMaxDynamicSharedMemorySize, GM_LDS_BYTES));
        FA_HIP(hipFuncSetAttribute((const void *)qkv_gemm_kernel<false, 8>, hipFuncAttributeMaxDynamicSharedMemorySize, GM_LDS_BYTES));
        FA_HIP(hipFuncSetAttribute((const void *)qkv_gemm_kernel<true, 8>, hipFuncAttributeMaxDynamicSharedMemorySize, GM_LDS_BYTES));
        FA_HIP(hipFuncSetAttribute((const void *)qkv_gemm_kernel<false, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, GM_LDS_BYTES));
        FA_HIP(hipFuncSetAttribute((const void *)qkv_gemm_kernel<true, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, GM_LDS_BYTES));
        lds_allowed.store(true, std::memory_order_release);
    }
    FaLaunchScope scope(ctx, l.n_kv ? "fused_qkv_gemm_kernel" : "matmul_gemm_kernel", true);
    if (tiles_whole && ctx->gemm_variant != 1) {
        if (l.weight_bits == 16) FA_TRY(fa_tile::launch_f16(ctx, scope, shape, a, l.canonical));
        else if (l.weight_bits == 8) FA_TRY(fa_tile::launch_q8(ctx, scope, shape, a, l.canonical));
        else FA_TRY(fa_tile::launch_q4(ctx, scope, shape, a, l.canonical));
        return scope.finish();
    }
    const uint32_t grid = (uint32_t)n_wg * a.k_splits;
    if (l.weight_bits == 4) {
        if (l.canonical) scope.launch(qkv_gemm_kernel<true, 4>, dim3(grid), dim3(GM_NT), GM_LDS_BYTES, a);
        else scope.launch(qkv_gemm_kernel<false, 4>, dim3(grid), dim3(GM_NT), GM_LDS_BYTES, a);
    } else if (q8) {
        if (l.canonical) scope.launch(qkv_gemm_kernel<true, 8>, dim3(grid), dim3(GM_NT), GM_LDS_BYTES, a);
        else scope.launch(qkv_gemm_kernel<false, 8>, dim3(grid), dim3(GM_NT), GM_LDS_BYTES, a);
    } else {
        if (l.canonical) scope.launch(qkv_gemm_kernel<true, 16>, dim3(grid), dim3(GM_NT), GM_LDS_BYTES, a);
        else scope.launch(qkv_gemm_kernel<false, 16>, dim3(grid), dim3(GM_NT), GM_LDS_BYTES, a);
    }
    FA_TRY(scope.finish());
    if (a.k_splits > 1) {
        FaLaunchScope fin(ctx, "gemm_finish_kernel", true);
        fin.launch(gemm_finish_kernel, dim3(ceil_div_u32(l.m * ceil_div_u32(a.n_total, 8), 256)), dim3(256), 0, a);
        FA_TRY(fin.finish());
    }
    return FA_OK;
}

fa_status fa_launch_fused_qkv_gemm(fa_ctx *ctx, const FusedQkvLaunch &l) { return launch_gemm(ctx, l, nullptr); }

fa_status fa_launch_fused_qkv_gemm_rope(fa_ctx *ctx, const FusedQkvLaunch &l, const QkvRopeLaunch &r) { return launch_gemm(ctx, l, &r); }
