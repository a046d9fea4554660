// How a FusedQkv / MatMul launch is laid out on the panel kernel (fa_panel.h): plain host arithmetic, so that it can be checked for any
// number of compute units without a card.
#pragma once

#include <algorithm>
#include <cstdint>

namespace fa_panel {

// What the layout depends on: weight rows of all matrices, features, input rows.
struct Shape {
    uint32_t total_rows, k_dim, m, weight_bits;
    bool canonical, gamma, rope;
};

inline uint32_t plan_ceil_div(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

// Two workgroups per compute unit: rows of up to 1024 features, except where the registers do not allow it.
constexpr bool two_per_cu(uint32_t nt, uint32_t nc, uint32_t pk, bool rope) { return pk <= 2 && !(rope && nt == 2 && nc == 2); }

// Below this many input rows block-quantised weights are summed block by block.
constexpr uint32_t BLOCK_SUMS_BELOW = 12;

// The most 16-row tiles of weight rows that a workgroup with passes of 16 input rows holds in registers.
inline uint32_t most_tiles(const Shape &s, uint32_t pk) {
    if (pk <= 2 || s.m <= 8 || (s.weight_bits != 16 && s.m < BLOCK_SUMS_BELOW)) return 2;
    return pk <= 4 ? 3 : s.weight_bits == 16 ? 5 : 4;
}

// How a FusedQkv / MatMul launch runs on the panel kernel (fa_panel.h): 16-row tiles of weight rows per workgroup, 16-row groups
// of input rows per pass, weight rows per workgroup, workgroups along the passes.
struct Plan {
    uint32_t nt, nc, pk, rows_per_wg, n_pass, grid_x, grid_y, rounds;
    bool eights = false;  // passes of 8 input rows
    uint32_t beside;  // grid_y where the workgroups of the same weight rows lie side by side on an XCD, else 0
};
// Whether the kernels have a form for the plan.
inline bool has_kernel(const Shape &s, const Plan &p) {
    return p.pk >= 1 && p.pk <= 6 && p.nt >= 1 && p.nt <= (p.eights || p.nc == 2 ? 2u : most_tiles(s, p.pk)) && p.rows_per_wg <= 16 * p.nt && p.nc >= 1 &&
           p.nc <= (p.pk <= 4 && !p.eights ? 2u : 1u) && !(p.eights && p.pk > 4);
}

inline Plan panel_plan(const Shape &s, uint32_t n_cus) {
    Plan p;
    p.pk = plan_ceil_div(s.k_dim, 512), p.nc = s.m <= 16 || p.pk > 4 ? 1u : 2u, p.n_pass = plan_ceil_div(s.m, 16 * p.nc);
    // Weight rows per workgroup: what a pass costs is mostly its input rows, whatever the weight rows, so as few passes as
    // possible on a compute unit - one after the other or, in two workgroups, side by side (Qwen2.5-0.5B, 64 rows: o_proj as 448
    // workgroups of 4 weight rows 5.2 us, as 112 of 16 3.9); of equal choices the fewest weight rows. A second tile of weight rows
    // costs a fifth of a pass, four fifths where the rows of F16 and Q8_0 weights are K apart and nothing is normalised (180 rows,
    // 896 x 896: 4.9 us as 336 workgroups of 16, 5.1 as 168 of 32), and a pass with its norm a fifth more beside another.
    uint64_t best = ~0ull;
    const uint32_t least = plan_ceil_div(s.total_rows, n_cus) < 32 ? (plan_ceil_div(s.total_rows, n_cus) + 1) & ~1u : 32u;
    for (uint32_t rpw : {least, 16u, 32u}) {
        const uint32_t gx = plan_ceil_div(s.total_rows, rpw), nt = rpw > 16 ? 2u : 1u;
        const bool two = two_per_cu(nt, p.nc, p.pk, s.rope);
        const uint32_t slots = two ? 2 * n_cus : n_cus;
        uint32_t gy = slots / gx;
        gy = gy < 1 ? 1u : gy > p.n_pass ? p.n_pass : gy;
        const uint32_t load = two ? std::max(gx * gy, n_cus) : plan_ceil_div(gx * gy, n_cus) * n_cus;
        const uint32_t tiles = nt == 1 ? 50u : !s.canonical && s.weight_bits != 4 && !s.gamma ? 90u : 60u;
        const uint32_t beside = two && gx * gy > n_cus && s.gamma ? 12u : 10u;
        const uint64_t cost = (uint64_t)load * plan_ceil_div(p.n_pass, gy) * tiles * beside;
        if (cost < best) best = cost, p.nt = nt, p.rows_per_wg = rpw, p.grid_x = gx, p.grid_y = gy, p.rounds = plan_ceil_div(gx * gy, slots);
    }
    // Rows of more than 2048 features: a workgroup per pass, with as many weight rows as put all of them in one round of workgroups. (One
    // workgroup for both passes, 20 weight rows: the second pass's rows are asked for, normalised and multiplied behind the first's. FusedQkv of
    // 5120 x 3072, 32 rows, F16 14.5 -> 11.5 us, Q8_0 14.3 -> 10.7, Q4_0 13.7 -> 10.6; 64 rows F16 19.3 -> 15.5; o_proj of 3072 x 3072,
    // 32 rows F16 8.1 -> 7.4, 48 rows 10.0 -> 7.7, Q8_0 10.0 -> 7.5.) The workgroups of the same weight rows are next to each other on an
    // XCD, so that memory is read once.
    // Shorter rows of 17 to 64 input rows (96 with a gamma, of up to 1024 features) likewise, 16 to a workgroup instead of 32, while up to two tiles of weight rows (three of more than
    // 1024 features) reach: half of the norm, which every workgroup works out for itself, for twice the weight rows. With a gamma always -
    // 32 rows of 1152 x 896 F16 5.4 -> 4.4 us, Q8_0 5.6 -> 4.5, of 2560 x 2048 8.3 -> 7.5, 8.1 -> 7.3, 48 rows 9.3 -> 7.8, 9.1 -> 7.1, 64 rows
    // 9.6 -> 8.7, 9.2 -> 8.2, 80 rows of 1152 x 896 F16 5.4 -> 5.0; but for the rotation of Q8_0 in two tiles of two pieces, 5.25 -> 5.46 -, without one where one tile reaches or the
    // other way has more than one round of passes: 32 rows of 896 x 896 F16 4.1 -> 3.4, of 2048 x 2048 5.9 -> 5.0, Q8_0 5.5 -> 4.5, 45 rows of 2240
    // x 2048 Q4_0 6.3 -> 5.3; beyond the lines 27 rows of 2688 x 2048 Q4_0 5.2 -> 5.4, 39 of 2048 x 2048 4.6 -> 5.4.
    const uint32_t passes = plan_ceil_div(s.m, 16);
    const bool wide = p.pk > 4;
    if (passes > 1 && (wide || passes <= (s.gamma && p.pk <= 2 ? 6u : 4u))) {
        const uint32_t groups = n_cus / (8 * passes) * 8, rows = (plan_ceil_div(s.total_rows, groups ? groups : 8) + 1) & ~1u;
        const uint32_t most = 16 * most_tiles(s, p.pk);
        const bool ahead = s.gamma ? !(s.rope && s.weight_bits == 8 && p.pk <= 2 && rows > 16 && passes >= 4)
                                   : rows <= 16 || (passes == 3 ? s.total_rows > 8 * n_cus && rows <= 40 : rows > 32);
        if (wide || (rows <= most && ahead)) {
            p.nc = 1, p.n_pass = passes, p.rows_per_wg = rows < most ? rows : most, p.nt = plan_ceil_div(p.rows_per_wg, 16);
            p.grid_x = plan_ceil_div(s.total_rows, p.rows_per_wg), p.grid_y = passes;
            p.rounds = plan_ceil_div(plan_ceil_div(p.grid_x, 8) * 8 * passes, n_cus);
        }
    }
    // 9 to 24 rows of up to 2048 features: 8 to a workgroup where that takes no more tiles of weight rows - with a gamma, or 9 to 16 rows
    // (F16: of up to 1024 features). us, 16 rows to a workgroup -> 8: 1152 x 896 with a gamma 16 rows F16 4.3 -> 3.9, Q8_0 4.4 -> 4.1, 24 rows
    // 4.3 -> 3.7, Q4_0 4.5 -> 3.8; 2560 x 2048 24 rows F16 7.4 -> 7.0, Q8_0 7.2 -> 6.3, Q4_0 7.0 -> 6.0; without one 2048 x 2048 16 rows Q4_0 4.4 ->
    // 4.0, 896 x 896 F16 3.4 -> 3.25. With a tile more 16 rows of 2560 x 2048 F16 6.3 -> 6.6, without a gamma 24 rows of 2048 x 2048 4.9 -> 5.9.
    const uint32_t eights = plan_ceil_div(s.m, 8);
    if (!wide && p.nc == 1 && (eights == 2 || (eights == 3 && s.gamma)) && (s.gamma || p.pk <= 2 || s.weight_bits != 16)) {
        const uint32_t groups = n_cus / (8 * eights) * 8, rows = (plan_ceil_div(s.total_rows, groups ? groups : 8) + 1) & ~1u;
        if (rows <= 16 * std::min(p.nt, 2u)) {
            p.eights = true, p.n_pass = p.grid_y = eights, p.rows_per_wg = rows, p.grid_x = plan_ceil_div(s.total_rows, rows), p.rounds = 1;
            p.nt = plan_ceil_div(rows, 16);
        }
    }
    p.beside = wide || (p.nc == 1 && p.n_pass > 1 && p.grid_y == p.n_pass) ? p.n_pass : 0;
    return p;
}

}  // namespace fa_panel
