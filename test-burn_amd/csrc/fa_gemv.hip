// FusedQkv and MatMul of ONE input row (a decode step): the weight stream without the matrix cores.
// Reference: the same ops as fa_qkv.hip - src/metals/gemv/qkv_step.rs:14-120, src/metals/gemv/qkv_project.metal,
// src/metals/rmsnorm/rmsnorm.metal:17-96, write stage src/metals/gemv/stages.rs:200-224.
//
// What bounds such a launch is the chain of instructions of one wave, not a unit: 256 workgroups of 512 threads that load an
// input row and 16 bytes of weights per thread, meet at two barriers and store take 1.98 us in a graph (an empty launch 1.6),
// while the kernel of fa_qkv.hip, which prepares for 16 input rows, took 4.1 to 4.9 us on 1 MB of weights. So everything that
// one row does not need is left out here: no 16-row tiles (their unused rows were loaded and multiplied all the same), no input
// row in LDS (a wave keeps the slice it multiplies in registers), two-way dot products instead of matrix instructions, scalar
// addressing, one barrier for the norm and one for the sums.
//
//   * rows are taken in groups of RL = 4 / 4 / 8 (F16 / Q8_0 / Q4_0). A lane owns 16 bytes of one row's 32-feature block:
//     lane = (block of KPL = 4 / 8 / 8, row of RL, part), so a request of a wave covers whole lines: in the canonical layout
//     KPL runs of 256 / 128 / 128 bytes (F16 with 128-byte runs, two rows: 88.8 us against 85.0 for four layers of the
//     Llama-3.2-3B block), in row-major weights RL runs;
//   * wave w takes the blocks KPL U w .. of every group, U requests each; the workgroup takes T groups, all U * T requests of a
//     lane in flight at once, groups fastest (consecutive groups are neighbours in the canonical layout);
//   * the lanes of a row are added with lane exchanges, the waves through LDS in wave order.
// Arithmetic as in fa_qkv.hip: the input normalised in f32 and rounded to f16, f32 sums, block scales applied to f32 block
// sums, one rounding at the end.
#include "fa_internal.h"
#include "fa_norm.h"
#include "fa_quant.h"
#include <type_traits>

namespace {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u4_t __attribute__((ext_vector_type(4)));

constexpr int GV_MAX_NW = 8;
constexpr int GV_RL_SHIFT(int wb) { return wb == 4 ? 3 : 2; }

struct GemvDev {
    const unsigned char *w[3];
    const __half *scales[3];
    const __half *x, *gamma, *residual;
    const __half *bias[3];
    __half *out[3];
    uint32_t rows0, rows1;          // rows of W_q and of W_k = W_v (0: one matrix)
    uint32_t groups0, groups1, n_groups;  // the same in groups of RL rows, and all of them
    uint32_t k_dim, nkb;
    uint32_t row_stride, kb_stride0, kb_stride1;  // bytes from row to row and from block to block (per row count)
    uint32_t n_waves;
    float eps, inv_k, alpha, beta;
};

__device__ __forceinline__ float dot8(h8_t a, h8_t b, float acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_fdot2(h2_t{a[2 * i], a[2 * i + 1]}, h2_t{b[2 * i], b[2 * i + 1]}, acc, false);
    return acc;
}

template <int WB, int U, int T>
__global__ void __launch_bounds__(64 * GV_MAX_NW, 2) gemv_row_kernel(GemvDev a_by_value) {
    static_assert(std::is_trivially_copyable<GemvDev>::value, "read as raw bytes from the argument block, where it is the first member");
    const GemvDev &a = *(const GemvDev *)__builtin_amdgcn_kernarg_segment_ptr();
    (void)a_by_value;
    constexpr int PARTS = WB == 16 ? 4 : WB == 8 ? 2 : 1, PARTS_SHIFT = WB == 16 ? 2 : WB == 8 ? 1 : 0, RL_SHIFT = GV_RL_SHIFT(WB), RL = 1 << RL_SHIFT, KPL = 64 / (PARTS * RL), E = 32 / PARTS;
    constexpr int XP = E / 8;  // 16-byte pieces of the input per unit
    __shared__ float red[GV_MAX_NW][RL * T];
    __shared__ float ss_lds[GV_MAX_NW];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
    const __half *const x = a.x, *const gamma = a.gamma;
    const uint32_t groups0 = a.groups0, groups1 = a.groups1, n_groups = a.n_groups, nkb = a.nkb, row_stride = a.row_stride;
    const uint32_t kb_stride0 = a.kb_stride0, kb_stride1 = a.kb_stride1, n_waves = a.n_waves;
    const unsigned char *const w0 = a.w[0], *const w1 = a.w[1], *const w2 = a.w[2];
    const __half *const s0 = a.scales[0], *const s1 = a.scales[1], *const s2 = a.scales[2];
    asm volatile("" ::"s"(x), "s"(gamma), "s"(groups0), "s"(groups1), "s"(n_groups), "s"(nkb), "s"(row_stride), "s"(kb_stride0), "s"(kb_stride1),
                 "s"(n_waves), "s"(w0), "s"(w1), "s"(w2));
    if constexpr (WB != 16) asm volatile("" ::"s"(s0), "s"(s1), "s"(s2));

    // The sums of the waves that a workgroup has not: -0, which adds nothing to any of the others. (So that all eight are asked for at
    // once: a loop over the waves there are was a trip to LDS for each, with a norm twice. FusedQkv of 1152 x 896 Q8_0 3.15 -> 2.93 us, F16
    // 3.42 -> 3.10, 5120 x 3072 F16 8.1 -> 7.7, Q8_0 7.7 -> 7.2, 2560 x 2048 Q8_0, all eight waves there, 4.33 -> 4.26; o_proj of 3072 5.78 -> 5.66.)
    for (uint32_t i = wave + n_waves; i < GV_MAX_NW; i += n_waves) {
        if (lane < RL * T) red[i][lane] = -0.0f;
        if (lane == 0) ss_lds[i] = -0.0f;
    }
    const uint32_t part = lane & (PARTS - 1), rsub = (lane >> PARTS_SHIFT) & (RL - 1), kbl = lane >> (PARTS_SHIFT + RL_SHIFT);
    // the lane's slice of the input row and of the norm's weights
    uint32_t kb[U];
    bool kb_ok[U];
    h8_t xv[U][XP], gv[U][XP];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t b = (wave * U + u) * KPL + kbl;
        kb_ok[u] = b < nkb, kb[u] = min(b, nkb - 1);
        const uint32_t off = kb[u] * 64 + part * (E * 2);
#pragma unroll
        for (int p = 0; p < XP; ++p) {
            xv[u][p] = *reinterpret_cast<const h8_t *>(reinterpret_cast<const unsigned char *>(x) + off + p * 16);
            gv[u][p] = fa_norm::load_global<h8_t>(reinterpret_cast<const unsigned char *>(gamma ? gamma : x) + off + p * 16);
        }
    }
    // every weight of the workgroup; a group past the last re-reads the last (its sums are not stored)
    const uint32_t g0 = blockIdx.x * T;
    u4_t wv[T][U];
    _Float16 sc[T][U];
    const unsigned char *base[T];
    const __half *sbase[T];
    uint32_t kbs[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        uint32_t g = min(g0 + t, n_groups - 1);
        base[t] = w0, sbase[t] = s0, kbs[t] = kb_stride0;
        if (g >= groups0) {
            g -= groups0, base[t] = w1, sbase[t] = s1, kbs[t] = kb_stride1;
            if (g >= groups1) g -= groups1, base[t] = w2, sbase[t] = s2;
        }
        base[t] += (size_t)g * RL * row_stride;
        if constexpr (WB != 16) sbase[t] += (size_t)g * RL * nkb;
    }
    // (groups fastest: in the canonical layout the lines of consecutive groups lie next to each other)
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < T; ++t)
            wv[t][u] = fa_norm::load_global_once<u4_t>(base[t] + (rsub * row_stride + kb[u] * kbs[t] + part * 16));
    if constexpr (WB != 16) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int t = 0; t < T; ++t)
                sc[t][u] = fa_norm::load_global<_Float16>(reinterpret_cast<const unsigned char *>(sbase[t]) + (rsub * nkb + kb[u]) * 2);
    }
    // what the thread that stores row tid of the workgroup adds to its sum
    const uint32_t rows0 = a.rows0, rows1 = a.rows1;
    const __half *const residual = a.residual;
    const __half *const b0 = a.bias[0], *const b1 = a.bias[1], *const b2 = a.bias[2];
    __half *const o0 = a.out[0], *const o1 = a.out[1], *const o2 = a.out[2];
    const float eps = a.eps, inv_k = a.inv_k, alpha = a.alpha, beta = a.beta;
    asm volatile("" ::"s"(rows0), "s"(rows1), "s"(residual), "s"(b0), "s"(b1), "s"(b2), "s"(o0), "s"(o1), "s"(o2), "s"(eps), "s"(inv_k), "s"(alpha), "s"(beta));
    const uint32_t gr = g0 * RL + min(tid, (uint32_t)(RL * T - 1));
    const bool store = tid < RL * T && gr < n_groups * RL;
    const __half *bp = b0;
    __half *op = o0;
    uint32_t lrow = min(gr, n_groups * RL - 1);
    if (lrow >= rows0) {
        lrow -= rows0, bp = b1, op = o1;
        if (lrow >= rows1) lrow -= rows1, bp = b2, op = o2;
    }
    const _Float16 bias = fa_norm::load_global<_Float16>(b0 ? bp + lrow : x);
    const _Float16 res = fa_norm::load_global<_Float16>(residual ? residual + lrow : x);

    if (gamma) {
        float ss = 0.0f;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int p = 0; p < XP; ++p) {
                const float q = dot8(xv[u][p], xv[u][p], 0.0f);
                ss += kb_ok[u] ? q : 0.0f;
            }
        ss = fa_norm::wave_sum(ss);  // (every feature RL times: once per row of the group)
        if (lane == 0) ss_lds[wave] = ss;
        __syncthreads();
        float tot = 0.0f;
#pragma unroll
        for (int i = 0; i < GV_MAX_NW; ++i) tot += ss_lds[i];
        const float inv_rms = fa_norm::inv_rms(tot, inv_k * (1.0f / RL), eps);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int p = 0; p < XP; ++p) xv[u][p] = fa_norm::scale8(xv[u][p], inv_rms, gv[u][p]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (!kb_ok[u]) {
#pragma unroll
            for (int p = 0; p < XP; ++p) xv[u][p] = h8_t{0, 0, 0, 0, 0, 0, 0, 0};
        }

    float acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        acc[t] = 0.0f;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const u4_t w = wv[t][u];
            if constexpr (WB == 16) {  // (past the last block the sum is left as it is: a product with the re-read weights is NaN where one is infinite)
                const float s = dot8(__builtin_bit_cast(h8_t, w), xv[u][0], acc[t]);
                acc[t] = kb_ok[u] ? s : acc[t];
            } else {
                float s;
                if constexpr (WB == 8) {
                    s = dot8(fa_quant::q8_to_f16<true>(w[0], w[1]), xv[u][0], 0.0f);
                    s = dot8(fa_quant::q8_to_f16<true>(w[2], w[3]), xv[u][1], s);
                } else {
                    s = 0.0f;
#pragma unroll
                    for (int q = 0; q < 4; ++q) s = dot8(fa_quant::q4_to_f16(w[q]), xv[u][q], s);
                }
                acc[t] += s * (kb_ok[u] ? (float)sc[t][u] : 0.0f);
            }
        }
    }
    // the lanes of a row: parts, then blocks
#pragma unroll
    for (int t = 0; t < T; ++t) {
        float v = acc[t];
        if constexpr (PARTS >= 2) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, true));  // quad_perm 1 0 3 2
        if constexpr (PARTS >= 4) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4e, 0xf, 0xf, true));  // quad_perm 2 3 0 1
        if constexpr (KPL >= 8) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, true));                           // row_ror:8
        acc[t] = fa_norm::sum_rows_of_16(v);
    }
    if (part == 0 && kbl == 0) {
#pragma unroll
        for (int t = 0; t < T; ++t) red[wave][t * RL + rsub] = acc[t];
    }
    __syncthreads();
    if (store) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < GV_MAX_NW; ++i) s += red[i][tid];
        s *= alpha;
        if (b0) s += (float)bias;
        if (residual) s += beta * (float)res;
        fa_norm::store_global(op + lrow, (_Float16)s);
    }
}

template <int WB, int U>
void launch_t(FaLaunchScope &scope, uint32_t t, dim3 grid, dim3 block, const GemvDev &a) {
    if (t == 1) scope.launch(gemv_row_kernel<WB, U, 1>, grid, block, 0, a);
    else if (t == 2) scope.launch(gemv_row_kernel<WB, U, 2>, grid, block, 0, a);
    else scope.launch(gemv_row_kernel<WB, U, 3>, grid, block, 0, a);
}

template <int WB>
void launch_u(FaLaunchScope &scope, uint32_t u, uint32_t t, dim3 grid, dim3 block, const GemvDev &a) {
    if (u == 1) launch_t<WB, 1>(scope, t, grid, block, a);
    else if (u == 2) launch_t<WB, 2>(scope, t, grid, block, a);
    else launch_t<WB, 4>(scope, t, grid, block, a);
}

}  // namespace

// Takes a launch of one input row: rows of every matrix in whole groups, up to 8192 features (what eight waves of four units
// hold) and matrices below 2 GiB (32-bit offsets); anything else stays with the kernel for up to 16 rows.
fa_status fa_launch_gemv_row(fa_ctx *ctx, const FusedQkvLaunch &l, bool *taken) {
    *taken = false;
    const uint32_t rl = 1u << GV_RL_SHIFT(l.weight_bits), kpl = l.weight_bits == 16 ? 4u : 8u, nkb = l.k_dim / 32;
    const uint64_t max_rows = l.n_dim > l.n_kv ? l.n_dim : l.n_kv;
    if (l.m != 1 || l.n_dim % rl != 0 || l.n_kv % rl != 0 || nkb > 32 * kpl || max_rows * l.k_dim * (uint32_t)l.weight_bits / 8 >= (1ull << 31)) return FA_OK;
    GemvDev a;
    memset(&a, 0, sizeof(a));
    for (int i = 0; i < 3; ++i)
        a.w[i] = reinterpret_cast<const unsigned char *>(l.w[i]), a.scales[i] = l.scales[i], a.bias[i] = l.bias[i], a.out[i] = l.out[i];
    a.x = l.x, a.gamma = l.gamma, a.residual = l.residual;
    a.rows0 = l.n_dim, a.rows1 = l.n_kv;
    a.groups0 = l.n_dim / rl, a.groups1 = l.n_kv / rl, a.n_groups = a.groups0 + 2 * a.groups1;
    a.k_dim = l.k_dim, a.nkb = nkb;
    const uint32_t blk = 4u * (uint32_t)l.weight_bits;  // bytes of a 32-feature block of one row
    a.row_stride = l.canonical ? blk : nkb * blk;
    a.kb_stride0 = l.canonical ? l.n_dim * blk : blk, a.kb_stride1 = l.canonical ? l.n_kv * blk : blk;
    a.eps = l.eps, a.inv_k = 1.0f / (float)l.k_dim, a.alpha = l.alpha, a.beta = l.beta;
    const uint32_t u = nkb <= 8 * kpl ? 1u : nkb <= 16 * kpl ? 2u : 4u;
    a.n_waves = ceil_div_u32(nkb, kpl * u);
    // Groups per workgroup: as few as leave at most two workgroups per compute unit, up to three (longer chains of one wave
    // cost more than more waves: Llama-3.2-3B Q8_0 block 83 / 82 / 80 / 85 / 84 us with 1 / 2 / 3 / 4 / 6, Qwen2.5-0.5B
    // 281 / 285 / 294 / 300 / 323).
    const uint32_t n_cus = ctx->n_cus > 0 ? (uint32_t)ctx->n_cus : 256u;
    uint32_t t = ceil_div_u32(a.n_groups, 2 * n_cus);
    if (t > 3) t = 3;
    FaLaunchScope scope(ctx, l.n_kv ? "fused_qkv_kernel" : "matmul_gemv_kernel", true);
    const dim3 grid(ceil_div_u32(a.n_groups, t)), block(64 * a.n_waves);
    if (l.weight_bits == 16) launch_u<16>(scope, u, t, grid, block, a);
    else if (l.weight_bits == 8) launch_u<8>(scope, u, t, grid, block, a);
    else launch_u<4>(scope, u, t, grid, block, a);
    *taken = true;
    return scope.finish();
}
