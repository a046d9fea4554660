"""The layout of FusedQkv / MatMul launches on the panel kernel (fa_panel_plan.h), for cards of any number of compute units: every
layout has a kernel, and its workgroups take every weight row with every pass of input rows, each once. The header is built for the CPU."""
import os
import subprocess

import foundry_attn as fa

SRC = r"""
#include <stdio.h>
#include <vector>
#include "fa_panel_plan.h"
using namespace fa_panel;
static unsigned long long plans, bad;
static void check(const Shape &s, uint32_t n_cus) {
    const Plan p = panel_plan(s, n_cus);
    bool ok = has_kernel(s, p);
    // as the kernel finds them (panel_kernel): weight rows from `along`, passes from `first` on
    const uint32_t pass_rows = p.form == EIGHTS ? 8 : 16 * p.nc, groups = (p.grid_x + 7) / 8 * 8, beside = p.beside();
    ok = ok && (unsigned long long)p.n_pass * pass_rows >= s.m && (p.n_pass - 1) * pass_rows < s.m;
    ok = ok && (unsigned long long)p.grid_x * p.rows_per_wg >= s.total_rows && (!s.rope || p.rows_per_wg % 2 == 0);
    if (ok && beside) {
        ok = p.workgroups() == groups * beside;
        std::vector<uint32_t> taken((size_t)groups * p.n_pass, 0);
        for (uint32_t id = 0; id < groups * beside; ++id) {
            const uint32_t eighth = id >> 3, group = eighth / beside, along = group * 8 + (id & 7), first = eighth - group * beside;
            for (uint32_t pass = first; pass < p.n_pass; pass += beside) ++taken[(size_t)along * p.n_pass + pass];
        }
        for (uint32_t t : taken) ok = ok && t == 1;
    } else if (ok) {
        ok = p.grid_y >= 1 && p.grid_y <= p.n_pass && p.workgroups() == p.grid_x * p.grid_y;
    }
    ++plans;
    if (!ok && ++bad <= 20)
        printf("%u CUs: %u rows x %u features, %u input rows, %u bits%s%s%s: %u tiles of %u rows, %u passes\n", n_cus, s.total_rows, s.k_dim, s.m,
               s.weight_bits, s.canonical ? "" : " row-major", s.gamma ? " gamma" : "", s.rope ? " rope" : "", p.nt, p.rows_per_wg, p.n_pass);
}
// what tests of test_gpu_panel.py are about: form and tiles on 256 compute units
static void expect(uint32_t rows, uint32_t k, uint32_t m, uint32_t bits, int canonical, int gamma, int rope, Form form, uint32_t nt) {
    const Plan p = panel_plan(Shape{rows, k, m, bits, canonical != 0, gamma != 0, rope != 0}, 256);
    if (p.form == form && p.nt == nt) return;
    ++bad;
    printf("%u rows x %u features, %u input rows, %u bits%s: form %d of %u tiles, not %d of %u\n", rows, k, m, bits, canonical ? "" : " row-major", p.form, p.nt, form, nt);
}
int main() {
    expect(5144, 2592, 40, 16, 0, 1, 0, WALK, 2), expect(4104, 2592, 40, 16, 0, 0, 0, WALK, 2), expect(3000, 2592, 40, 16, 0, 0, 0, WALK, 1);
    expect(5144, 2592, 40, 8, 0, 1, 0, WALK, 2), expect(5144, 2592, 33, 4, 1, 1, 0, WALK, 2);
    expect(1288, 2592, 35, 8, 0, 1, 0, WALK, 1), expect(408, 2592, 20, 4, 1, 1, 0, WALK, 1);
    expect(5376, 2592, 33, 16, 0, 1, 1, WALK, 2), expect(3840, 2592, 40, 16, 0, 0, 1, WALK, 1);
    for (uint32_t bits : {8u, 4u}) expect(5376, 2592, 33, bits, bits == 8, 1, 1, WALK, 2), expect(1344, 2592, 35, bits, 1, 1, 1, WALK, 1);
    for (uint32_t bits : {16u, 8u, 4u}) {
        expect(5152, 2112, 17, bits, 0, 1, 0, BESIDE, 3), expect(8096, 3072, 18, bits, 1, 1, 0, BESIDE, 4);
        expect(5120, 3072, 32, bits, 1, 1, 1, BESIDE, 3), expect(5120, 3072, 40, bits, 1, 1, 1, BESIDE, 4);
        expect(3072, 2048, 64, bits, 0, 1, 0, bits == 8 ? WALK : BESIDE, bits == 8 ? 2 : 3), expect(3072, 1984, 64, bits, 0, 1, 0, BESIDE, 3);
        expect(896, 896, 32, bits, 1, 0, 0, BESIDE, 1), expect(1152, 896, 16, bits, 1, 1, 0, EIGHTS, 1), expect(2560, 2048, 24, bits, 1, 1, 1, EIGHTS, 2);
        expect(2560, 2048, 24, bits, 0, 1, 1, bits == 4 ? EIGHTS : WALK, bits == 4 ? 2 : 1);
    }
    expect(5120, 2592, 64, 16, 1, 1, 0, BESIDE, 5), expect(5120, 3072, 64, 16, 1, 1, 1, BESIDE, 5), expect(4864, 2592, 57, 16, 1, 1, 1, BESIDE, 5), expect(5120, 3072, 57, 16, 1, 1, 1, BESIDE, 5);
    for (uint32_t n_cus = 8; n_cus <= 320; n_cus += n_cus < 64 ? 4 : 8)
        for (uint32_t bits : {4u, 8u, 16u})
            for (int flags = 0; flags < 8; ++flags)
                for (uint32_t k : {64u, 512u, 544u, 1024u, 1056u, 2048u, 2080u, 3072u})
                    for (uint32_t m : {2u, 8u, 9u, 11u, 12u, 16u, 17u, 24u, 25u, 32u, 33u, 48u, 49u, 64u, 65u, 96u, 128u, 416u})
                        for (uint32_t rows : {2u, 64u, 770u, 1152u, 1904u, 2560u, 4098u, 5120u, 8192u, 10600u, 40000u})
                            check(Shape{rows, k, m, bits, (flags & 1) != 0, (flags & 2) != 0, (flags & 4) != 0}, n_cus);
    printf("%llu layouts, %llu bad\n", plans, bad);
    return bad != 0;
}
"""


def test_every_layout_has_a_kernel(tmp_path):
    src, exe = tmp_path / "plan.cpp", str(tmp_path / "plan")
    src.write_text(SRC)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-I", os.path.join(os.path.dirname(fa.__file__), "csrc"), str(src), "-o", exe])
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
