// FusedQkv and MatMul of a chunk of input rows that fits a workgroup's LDS 32 rows at a time ("panel"): one launch, RMSNorm and
// KvPrepFused included. Reference: the same ops as fa_qkv.hip and fa_gemm.hip - src/metals/gemv/qkv_step.rs:14-120,
// src/metals/matmul.rs:190-239, src/metals/rmsnorm/rmsnorm.metal:17-96, write stage src/metals/gemv/stages.rs:200-224,
// src/metals/kv_prep/kv_prep_fused.metal:45-122.
//
// A chunk of a few dozen rows (a default prefill chunk of 32, a server's batch of sequences) is still a weight stream, but every
// compute unit needs all of its input rows, normalised. What that costs is how they are asked for: a request in the layout of
// the matrix instruction's operand (16 rows x 64 bytes, one row per lane of a 16-lane group) moves 37 KB/us into a compute unit
// from L2, a request along a row 108 to 130 KB/us. So rows are fetched along themselves, whole rows per wave (row r by wave
// r % 8), normalised in the registers they arrive in (no exchange between waves), written to LDS and read back as operands:
//   * a workgroup (8 waves) owns one or more 16-row tiles of weight rows. Its passes of input rows are divided in one of three forms, chosen
//     in fa_panel_plan.h:
//       - WALK: up to two tiles and passes of 32 input rows (16 of more than 2048 features), which it goes through one after the other. All its
//         weights are requested once, straight into the operand layout, behind the first pass's input rows; a pass's rows are requested
//         while the one before is multiplied. Few weight rows and many input rows: the passes are spread over workgroups (grid y);
//       - BESIDE: one pass of 16 input rows and up to five tiles (two of up to 1024 features, three of up to 2048); the workgroups of the same
//         weight rows lie next to each other on an XCD. Of more than 2048 features a few requests of every tile are on their way at a
//         time (RING);
//       - EIGHTS: the same with passes of 8 rows and up to two tiles;
//   * wave w multiplies the feature blocks 16 j + 2 w and 16 j + 2 w + 1 of every 512 features (adjacent: the two requests touch
//     the same lines);
//   * the eight waves' partial tiles meet in LDS and are added in wave order; then alpha, bias, beta * residual and one
//     rounding, or the KvPrepFused work on the rounded values (a workgroup then takes whole rotation pairs);
//   * NeoX pairs of a workgroup of up to 16 weight rows, and of the last of an odd number of tiles, lie in one tile, 8 rows from each half
//     (two tiles of which half the rows did not exist: 1152 x 896, 8 rows, F16 4.4 -> 3.8 us, Q8_0 4.9 -> 4.0, Q4_0 5.0 -> 4.1; 2560 x 2048
//     6.4 -> 5.4, 7.0 -> 5.4, 6.7 -> 5.2).
// Block-quantised weights become f16(weight * scale) as in the GEMM (src/metals/mma/tile_loader.metal:100-120); below 12 input
// rows (SUMS) they follow the weight stream: a matrix instruction covers one 32-feature block, its f32 sums times the scale.
#pragma once

#include <type_traits>

#include "fa_internal.h"
#include "fa_norm.h"
#include "fa_panel_plan.h"
#include "fa_qkv_rope.h"

namespace fa_panel {

constexpr int NTHREADS = 512, NW = NTHREADS / 64;

struct PanelDev {
    const unsigned char *w[3];
    const __half *scales[3], *bias[3];
    __half *out[3];
    uint32_t rows0, rows1, total_rows;  // of W_q, of W_k and W_v each, of all
    const __half *x, *gamma, *residual;
    uint32_t k_dim, m, rows_per_wg, canonical, n_pass;
    uint32_t beside, inv_beside;  // workgroups of the same weight rows on one XCD, side by side, and fa_inverse of it; 0: along grid y
    float eps, inv_k, alpha, beta;
    RopeDev r;
    uint32_t scale_pairs;  // a row holds an even number of scales, 4-byte aligned
    uint32_t block_shift;  // log2 of the page size, 32 = not a power of two
};

// A row in LDS: its 512-feature pieces, and 16 bytes so that 16 consecutive rows fall into 16 different bank groups.
template <int PK>
constexpr int row_bytes() { return PK * 1024 + 16; }
template <int NT, int NC>
constexpr int reduce_bytes() { return NW * NT * NC * 16 * 17 * 4; }
template <int PK>
constexpr bool G_IN_LDS = PK > 4;  // the longest rows: the norm's weights in LDS instead of registers
template <int PK>
constexpr int LDS_SHARE = (PK <= 2 ? 80 * 1024 : 160 * 1024) - 6 * 1024;  // two workgroups per compute unit, or one; less the scales
// Block-quantised weights: their scales as f16 [block][slot], with 8 bytes between blocks: a wave writes the blocks of two or three
// rows side by side, all of them to one bank without (o_proj of 1536 features x 4096 rows, 40 input rows: Q8_0 7.06 -> 6.64 us).
template <int NT>
constexpr int scale_stride() { return NT * 16 + 4; }
template <int NT, int PK>
constexpr int scale_bytes() { return scale_stride<NT>() * PK * 16 * 2; }
// The waves' sums get LDS of their own where it is there (a barrier less per pass), else they go over the rows.
template <int NT, int NC, int PK>
constexpr bool REDUCE_APART = NC * 16 * row_bytes<PK>() + reduce_bytes<NT, NC>() + (G_IN_LDS<PK> ? PK * 1024 : 0) + (NT > 3 ? scale_bytes<NT, PK>() : 0) <= LDS_SHARE<PK>;
template <int NT, int NC, int PK>
constexpr int lds_rows_bytes() {
    const int rows = NC * 16 * row_bytes<PK>(), red = reduce_bytes<NT, NC>();
    return REDUCE_APART<NT, NC, PK> ? rows + red : rows > red ? rows : red;
}
// Q4_0 with per-block sums, more than 1024 features: weights are fetched along memory and turned into operand order in LDS.
template <int WB, int PK, bool SUMS>
constexpr bool TURNS = WB == 4 && SUMS && PK > 2;
// Behind everything else, for that: room for each wave to turn weights into operand order, a KiB at a time.
template <int WB, int NT, int NC, int PK>
constexpr int turn_at() { return (lds_rows_bytes<NT, NC, PK>() + (G_IN_LDS<PK> ? PK * 1024 : 0) + (WB != 16 ? scale_bytes<NT, PK>() : 0) + 15) & ~15; }
template <int WB, int NT, int NC, int PK, bool SUMS>
constexpr int lds_bytes() { return turn_at<WB, NT, NC, PK>() + (TURNS<WB, PK, SUMS> ? NW * 1024 : 0); }

// launchers per weight width (one translation unit each)
template <int WB>
fa_status launch(FaLaunchScope &scope, bool rope, bool sums, const Plan &plan, const PanelDev &a);

}  // namespace fa_panel
