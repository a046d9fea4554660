// How a FusedQkv / MatMul launch is laid out on the panel kernel (fa_panel.h): plain host arithmetic, so that it can be checked for any
// card without one.
#pragma once

#include <algorithm>
#include <cstdint>

namespace fa_panel {

// What the layout depends on.
struct Shape {
    uint32_t total_rows, k_dim, m;  // weight rows of all matrices, features, input rows
    uint32_t weight_bits;
    bool canonical, gamma, rope;
};

// WALK: a workgroup takes passes of 16 or 32 input rows one after the other. BESIDE, EIGHTS: it has one pass, of 16 or 8 rows, and those of
// the same weight rows lie next to each other on an XCD.
enum Form { WALK, BESIDE, EIGHTS };

struct Plan {
    Form form;
    uint32_t nt, nc, pk;   // 16-row tiles of weight rows per workgroup, 16-row groups of input rows per pass, 512-feature pieces of a row
    uint32_t rows_per_wg;  // weight rows
    uint32_t n_pass, grid_x, grid_y, rounds;  // passes; workgroups along the weight rows and along the passes; rounds of workgroups
    bool ok;               // there is such a layout

    uint32_t beside() const { return form == WALK ? 0 : n_pass; }
    uint32_t workgroups() const { return form == WALK ? grid_x * grid_y : (grid_x + 7) / 8 * 8 * n_pass; }
};

// Two workgroups per compute unit: rows of up to 1024 features, except where the registers do not allow it.
constexpr bool two_per_cu(uint32_t nt, uint32_t nc, uint32_t pk, bool rope) { return pk <= 2 && !(rope && nt == 2 && nc == 2); }

// Below this many input rows block-quantised weights are summed block by block.
constexpr uint32_t BLOCK_SUMS_BELOW = 12;

// The most 16-row tiles of weight rows that a workgroup holds in registers.
inline uint32_t most_tiles(const Shape &s, Form form, uint32_t pk) {
    if (form != BESIDE || pk <= 2 || s.m <= 8 || (s.weight_bits != 16 && s.m < BLOCK_SUMS_BELOW)) return 2;
    return pk <= 4 ? 3 : s.weight_bits == 16 ? 5 : 4;
}

// Whether fa_panel::launch has a kernel for the plan.
inline bool has_kernel(const Shape &s, const Plan &p) {
    return p.ok && p.pk >= 1 && p.pk <= 6 && p.nt >= 1 && p.nt <= most_tiles(s, p.form, p.pk) && p.rows_per_wg <= 16 * p.nt && p.nc >= 1 &&
           p.nc <= (p.form == WALK && p.pk <= 4 ? 2u : 1u) && !(p.form == EIGHTS && p.pk > 4);
}

inline uint32_t plan_ceil_div(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

// Weight rows per workgroup: what a pass costs is mostly its input rows, whatever the weight rows, so as few passes as
// possible on a compute unit - one after the other or, in two workgroups, side by side (Qwen2.5-0.5B, 64 rows: o_proj as 448
// workgroups of 4 weight rows 5.2 us, as 112 of 16 3.9); of equal choices the fewest weight rows. A second tile of weight rows
// costs a fifth of a pass, four fifths where the rows of F16 and Q8_0 weights are K apart and nothing is normalised (180 rows,
// 896 x 896: 4.9 us as 336 workgroups of 16, 5.1 as 168 of 32), and a pass with its norm a fifth more beside another.
inline Plan walk_plan(const Shape &s, uint32_t n_cus) {
    Plan p{};
    p.ok = true, p.form = WALK;
    p.pk = plan_ceil_div(s.k_dim, 512), p.nc = s.m <= 16 || p.pk > 4 ? 1u : 2u, p.n_pass = plan_ceil_div(s.m, 16 * p.nc);
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
    // (of the longest rows, a workgroup with one pass has the kernel of those)
    if (p.pk > 4 && p.n_pass == 1) p.form = BESIDE;
    return p;
}

// A workgroup for each pass of 16 (8) input rows, with as many weight rows as put all of them in one round of workgroups.
inline Plan beside_plan(const Shape &s, uint32_t n_cus, Form form) {
    Plan p{};
    const uint32_t pass_rows = form == EIGHTS ? 8 : 16;
    p.form = form, p.pk = plan_ceil_div(s.k_dim, 512), p.nc = 1, p.n_pass = p.grid_y = plan_ceil_div(s.m, pass_rows);
    const uint32_t groups = n_cus / (8 * p.n_pass) * 8;
    if (groups == 0 || (form == EIGHTS && p.pk > 4)) return p;
    p.rows_per_wg = (plan_ceil_div(s.total_rows, groups) + 1) & ~1u, p.nt = plan_ceil_div(p.rows_per_wg, 16);
    p.grid_x = plan_ceil_div(s.total_rows, p.rows_per_wg), p.rounds = 1;
    p.ok = p.nt <= most_tiles(s, form, p.pk);
    return p;
}

// Whether a workgroup for each pass of 16 rows (`b`) is ahead of walking over them (`w`). It halves or quarters the chain of a workgroup -
// the rows that it fetches, normalises and multiplies -, for more weight rows to each: 0.72 to 0.91 of the time where those
// take no more tiles. With a tile more, what a workgroup asks for beside the rows decides. Time / walking of 5500 launches
// of 9 to 128 rows x 64 to 3072 features x 256 to 10500 weight rows, on one hardware queue, the other side of each line last:
//   up to 2048 features, a tile more
//     with a gamma, from 33 rows 0.92-0.99 (Q8_0 in three tiles, rows a multiple of 2 KB apart: 1.03), 25 to 32 rows 0.87-0.96 (F16 row-major
//       in two tiles of more than 1024 features: 1.02), 17 to 24 rows Q4_0 and canonical F16 of up to 1024 features 0.95-0.98, longer Q4_0 canonical or
//       in three tiles 0.92-0.96 (others 0.99-1.10);
//     without one 0.83-0.96 where walking gives a compute unit more than one pass, 0.92-0.97 in three tiles from 33 rows and Q4_0 canonical from
//       17 (with the rotation 1.01-1.11; others 1.02-1.10);
//   longer rows 0.76-0.98
//     F16 row-major, whose tiles ask for lines 16 rows apart: without a gamma where one round of workgroups walks over all passes 0.99-1.37
//       (27 of 28 launches; Q4_0 in four tiles there, two passes or one tile to walk with, 0.94-1.15, 1.06 in the mean), in five tiles over
//       three passes 1.05-1.11;
//     where walking has a workgroup for each pass: a tile more 1.04-1.17 (F16 in three tiles 0.77-0.87), Q4_0 canonical with up to 6 weight rows
//       1.01-1.04.
// (FusedQkv of 5120 x 3072, 32 rows, F16 14.5 -> 11.5 us, Q8_0 14.3 -> 10.7, Q4_0 13.7 -> 10.6; o_proj of 3072 x 3072 32 rows F16 8.1 -> 7.4, 48 rows
// Q8_0 10.0 -> 7.5; FusedQkv of 2560 x 2048 48 rows Q4_0 8.8 -> 6.9, of 1152 x 896 32 rows F16 5.4 -> 4.4.)
inline bool beside_ahead(const Shape &s, const Plan &w, const Plan &b, uint32_t n_cus) {
    const uint32_t passes = b.n_pass, walked = plan_ceil_div(w.n_pass, w.grid_y);
    if (!b.ok || passes < 2) return false;
    const bool f16 = s.weight_bits == 16, q8 = s.weight_bits == 8, q4 = s.weight_bits == 4, more_tiles = b.nt > w.nt;
    if (w.pk > 4) {
        if (walked == 1) return (!more_tiles && !(q4 && s.canonical && b.rows_per_wg <= 6)) || (f16 && b.nt == 3);
        const bool one_walks_all = w.grid_y == 1 && w.rounds == 1;
        if (f16 && !s.canonical) return s.gamma ? walked != 3 || b.nt < 5 : !one_walks_all;
        return !(q4 && !s.gamma && b.nt == 4 && one_walks_all && (w.nt == 1 || passes == 2));
    }
    if (passes > (s.gamma && w.pk <= 2 ? 6u : 4u)) return false;
    if (!more_tiles) return true;
    const bool rows_2k_apart = q8 && !s.canonical && s.k_dim % 2048 == 0;
    if (!s.gamma) return w.grid_x * w.grid_y * walked > n_cus || (b.nt == 3 && !s.rope && !rows_2k_apart && (passes > 2 || (q4 && s.canonical)));
    if (s.rope && q8 && w.pk <= 2 && passes >= 4) return false;  // (two tiles with the rotation: 5.25 -> 5.46 us)
    if (s.m <= 24) return w.pk <= 2 ? q4 || (f16 && s.canonical) : q4 && (s.canonical || b.nt == 3);
    if (s.m <= 32 && f16 && !s.canonical && w.pk > 2 && b.nt == 2) return false;
    return !(rows_2k_apart && b.nt == 3);
}

// Whether passes of 8 rows (`e`), of 9 to 24 rows of up to 2048 features, are ahead of that: with a gamma, or of 9 to 16 rows (F16: of up
// to 1024 features), where they take no more tiles - 0.68 to 0.98 of the walk, but for F16 row-major without a gamma, 0.99-1.07, and Q8_0 row-major with
// its blocks summed one by one, 1.04-1.12; of 17 to 24 rows with a gamma for a tile more, too - 0.85-0.90, F16 and Q8_0 row-major of more than 1024
// features 1.01. (9 to 16 rows for a tile more 1.02-1.35. 1152 x 896 with a gamma, 24 rows F16 4.3 -> 3.7 us, Q4_0 4.5 -> 3.8; 2560 x 2048 24 rows
// Q8_0 7.2 -> 6.3; without one 2048 x 2048 16 rows Q4_0 4.4 -> 4.0.)
inline bool eights_ahead(const Shape &s, const Plan &w, const Plan &b, const Plan &e) {
    if (!e.ok || s.m < 9 || s.m > (s.gamma ? 24u : 16u)) return false;
    if (!s.gamma && (s.weight_bits == 16 ? w.pk > 2 || !s.canonical : s.weight_bits == 8 && !s.canonical && w.pk > 2 && s.m < BLOCK_SUMS_BELOW)) return false;
    if (e.nt <= w.nt) return true;
    return s.m > 16 && (w.pk <= 2 || s.canonical || s.weight_bits == 4) && !(b.ok && b.nt <= w.nt);
}

// The layout of a launch.
inline Plan panel_plan(const Shape &s, uint32_t n_cus) {
    const Plan w = walk_plan(s, n_cus), b = beside_plan(s, n_cus, BESIDE), e = beside_plan(s, n_cus, EIGHTS);
    return eights_ahead(s, w, b, e) ? e : beside_ahead(s, w, b, n_cus) ? b : w;
}

}  // namespace fa_panel
