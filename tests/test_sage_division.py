"""The int8 quantiser divides a whole 32-row block by one f16 scale, a query's head by its f32 one. The kernels do the divisor's share of
an f32 division once (reciprocal estimate + one refinement) and per value one step to the quotient, a clamp and a rounding by addition
(fa_sage_quant.h). This builds that header for the CPU, the GPU's instructions put in by what they do, and checks its bytes against
clamp(rint(x / scale)): every positive finite f16 scale with numerators spread over many binades and within a few ulps of
(k + 1/2) * scale, the quantiser's rounding boundaries; every f16 value / 127 as a query's scale (one binade of them, the rest is the same up to
a power of two) with every f16 value of up to 13 binades below; scales that are zero, infinite or no number; the reciprocal estimate
exact and off by one ulp either way. Of a scale that is one, the quotients themselves have to be equal to the bit."""
import os
import subprocess

import foundry_attn as fa

HIP = r"""
#pragma once
#include <math.h>
#include <stdint.h>
#include <string.h>
#define __device__
#define __forceinline__ inline
extern int estimate_off;  /* ulps that the hardware's estimate is off */
static inline float ulps(float x, int d) { uint32_t u; memcpy(&u, &x, 4); u += (uint32_t)d; float y; memcpy(&y, &u, 4); return y; }
static inline float rcp(float d) { const float r = 1.0f / d; return r == 0.0f || isinf(r) || isnan(r) ? r : ulps(r, estimate_off); }
/* the middle one of three; the least of the others where the first is no number */
static inline float med3(float a, float lo, float hi) { return isnan(a) ? fminf(lo, hi) : fminf(fmaxf(a, lo), hi); }
static inline uint32_t perm(uint32_t a, uint32_t b, uint32_t s) {
    uint32_t o = 0;
    for (int i = 0; i < 4; ++i) {
        const uint32_t c = s >> 8 * i & 255;
        o |= (c > 7 ? 0u : (c > 3 ? a >> 8 * (c - 4) : b >> 8 * c) & 255) << 8 * i;
    }
    return o;
}
#define __builtin_amdgcn_rcpf rcp
#define __builtin_amdgcn_fmed3f med3
#define __builtin_amdgcn_perm perm
"""

SRC = r"""
#include <stdio.h>
#include <initializer_list>
#include "fa_sage_quant.h"
int estimate_off;
static unsigned long long bad, n;
static float f16_value(uint16_t h) {
    const uint32_t e = (h >> 10) & 31, m = h & 1023;
    return e == 0 ? ldexpf((float)m, -24) : ldexpf((float)(m + 1024), (int)e - 25);
}
static int wanted(float x, float d) {
    if (!(d > 0.0f)) return 0;
    const float q = rintf(x / d);
    return isnan(q) || q < -127.0f ? -127 : q > 127.0f ? 127 : (int)q;
}
static void check(const float (&x)[4], float d, bool equal_quotients) {
    const SageDivisor v = sage_divisor(d);
    const uint32_t got = sage_quant4_i8(x[0], x[1], x[2], x[3], v);
    for (int i = 0; i < 4; ++i) {
        const float q0 = x[i] * v.r, q = fmaf(fmaf(-v.d, q0, x[i]), v.r, q0);
        const bool same = !equal_quotients || q == x[i] / d;
        ++n;
        if ((int8_t)(got >> 8 * i) == wanted(x[i], d) && (int8_t)sage_quant_byte(x[i], v) == wanted(x[i], d) && same) continue;
        if (bad++ < 5) printf("d=%a x=%a got %d, %d (quotient %a)\n", d, x[i], (int8_t)(got >> 8 * i), wanted(x[i], d), q);
    }
}
int main(void) {
    uint32_t seed = 12345;
    const float inf = INFINITY, no = NAN;
    for (estimate_off = -1; estimate_off <= 1; ++estimate_off) {
        for (uint32_t h = 1; h < 0x7c00; ++h) {
            const float d = f16_value((uint16_t)h);
            for (int t = 0; t < 50; ++t) {
                float x[4];
                for (int i = 0; i < 4; ++i) {
                    seed = seed * 1664525u + 1013904223u; const uint32_t a = seed;
                    seed = seed * 1664525u + 1013904223u;
                    if (i & 1) x[i] = ulps(((float)((int)(a % 300) - 150) + 0.5f) * d, (int)(seed % 7) - 3);
                    else x[i] = ldexpf((float)(a >> 8) / 16777216.0f * 2.0f - 1.0f, (int)(seed % 40) - 30) * d * 256.0f;
                }
                check(x, d, true);
            }
            check({0.0f, -0.0f, no, 127.5f * d}, d, false);
        }
        for (int a = 1024; a < 2048; ++a)
            for (int e = 0; e < 14; ++e)
                for (int m = 1024; m < 2048; ++m) {
                    const float x = ldexpf((float)m, -e), d = (float)a / 127.0f;
                    if (x > (float)a) break;
                    check({x, -x, x, -x}, d, true);
                }
        for (float d : {0.0f, -0.0f, -1.0f, inf, -inf, no})
            for (float x : {0.0f, -0.0f, 1.0f, -65504.0f, 6e-8f}) {
                check({x, inf, -inf, no}, d, false);
                check({-x, x * 0.5f, x + 1.0f, x}, d, false);
            }
    }
    printf("checked %llu bad %llu\n", n, bad);
    return bad != 0;
}
"""


def test_quantised_bytes_are_those_of_the_division(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "t.cpp").write_text(SRC)
    csrc = os.path.join(os.path.dirname(os.path.abspath(fa.__file__)), "csrc")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-I", str(tmp_path), "-I", csrc, "-o", str(tmp_path / "t"), str(tmp_path / "t.cpp"), "-lm"], check=True)
    out = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout[-800:]
    assert "bad 0" in out.stdout and int(out.stdout.split()[1]) > 50_000_000
