"""GPU parity of the one-input-row weight stream (FusedQkv and MatMul at m = 1) where its split of the work ends: row groups that
do not fill a workgroup, workgroups across two matrices, feature blocks that do not fill the last wave's share, the longest
row it takes and rows past it. Against the oracle with the bars of test_gpu_qkv.py."""
import numpy as np
import pytest

import foundry_attn as fa
import orc
from gpu_util import announce, ctx
from test_gpu_qkv import _close, _data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K,N,NK", [
    (32, 8, 8),          # one block, one group per matrix
    (160, 40, 24),       # a workgroup's groups across the three matrices
    (672, 24, 8),        # six waves (block-quantised three): the sums of those that a workgroup has not
    (896, 16, 8),        # seven (four)
    (1056, 1544, 8),     # F16: one block past what eight waves of one unit hold; two groups per workgroup
    (2080, 4104, 16),    # the quantised forms: the same; three groups per workgroup, the last one partly filled
    (4096, 520, 520),    # F16: the longest row; the quantised forms: two units
    (4128, 64, 8),       # past F16's longest row (the kernel for up to 16 rows takes it)
    (8192, 48, 16),      # the quantised forms' longest row
])
def test_one_input_row(K, N, NK, weights, layout):
    announce("one input row", K, N, NK, weights, layout)
    f = ctx()
    rng = np.random.default_rng(K + N + NK)
    x, g, ws, bs = _data(rng, K, N, NK, 1)
    dx, dg, db = f.array(x), f.array(g), [f.array(b) for b in bs]
    outs = [f.zeros((1, n)) for n in (N, NK, NK)]
    res = rng.uniform(-1, 1, (1, N)).astype(np.float16)
    dres, dout = f.array(res), f.zeros((1, N))
    if weights == "f16":
        dev_w, scales, dev_s = [f.array(orc.to_canonical(w) if layout else w.reshape(-1)) for w in ws], None, []
        want = orc.fused_qkv(x, *ws, gamma=g, biases=bs, layout=0)
        want_mm = orc.matmul_gemv(x, ws[0], bs[0], res, 0, 32, 0.5, 0.75)
        arg = [w.arg() for w in dev_w]
    else:
        quant = [orc.quantize_q8_0(w) if weights == "q8" else orc.quantize_q4_0(w) for w in ws]
        dev_s = [f.array(s) for _, s in quant]
        scales = [s.arg() for s in dev_s]
        ints = [q for q, _ in quant]
        flat = [orc.to_canonical(q) if layout else q.reshape(-1) for q in ints]
        dev_w = [f.array(q if weights == "q8" else orc.pack_q4_0(q)) for q in flat]
        arg = [w.arg() if weights == "q8" else w.arg((n, K), dtype=fa.DTYPE_Q4_0) for w, n in zip(dev_w, (N, NK, NK))]
        want = orc.fused_qkv_q8(x, ints, [s for _, s in quant], gamma=g, biases=bs)
        want_mm = orc.matmul_gemv_q8(x, ints[0], quant[0][1], bs[0], res, 0, 32, 0.5, 0.75)
    f.fused_qkv(dx.arg(), *arg, *[o.arg() for o in outs], K, N, NK, 1, gamma=dg.arg(), biases=[b.arg() for b in db], layout=layout,
                scales=scales)
    f.matmul(dx.arg(), arg[0], dout.arg(), 1, N, K, bias=db[0].arg(), c=dres.arg(), transpose_b=not layout, alpha=0.5, beta=0.75,
             b_scales=scales[0] if scales else None)
    for o, w in zip(outs, want):
        got = o.download()
        assert np.all(np.isfinite(got)) and _close(got, w, K), float(np.max(np.abs(got.astype(np.float64) - w.astype(np.float64))))
    got, w = dout.download().astype(np.float64), want_mm.astype(np.float64)
    assert np.all(np.abs(got - w) <= 2 * np.maximum(np.abs(w), 2.0 ** -10) * 2.0 ** -10 + 1e-4), float(np.max(np.abs(got - w)))
    for b in [dx, dg, dres, dout] + db + outs + dev_w + dev_s:
        b.free()


def infinite_last_block(K, N, m, weights, layout):
    """MatMul whose weight row 1 is infinite in its last block (F16: one weight, block-quantised: the block's scale) under an input
    without negative values: the row's sums are infinite, every other row is the oracle's. What a kernel requests past the last block
    must not reach the sums."""
    f = ctx()
    rng = np.random.default_rng(K + N + m)
    x = rng.uniform(0.25, 1, (m, K)).astype(np.float16)
    w = rng.uniform(-0.1, 0.1, (N, K)).astype(np.float16)
    if weights == "f16":
        full = w.copy()
        w[1, K - 3] = np.inf
        dev_w, dev_s = f.array(orc.to_canonical(w) if layout else w.reshape(-1)), None
        arg = dev_w.arg()
    else:
        q, s = orc.quantize_q8_0(w) if weights == "q8" else orc.quantize_q4_0(w)
        full = orc.dequantize_blocks(q, s)
        q[1, K - 32:] = 3
        s[1, -1] = np.inf
        flat = orc.to_canonical(q) if layout else q.reshape(-1)
        dev_w, dev_s = f.array(flat if weights == "q8" else orc.pack_q4_0(flat)), f.array(s)
        arg = dev_w.arg() if weights == "q8" else dev_w.arg((N, K), dtype=fa.DTYPE_Q4_0)
    dx, dout = f.array(x), f.zeros((m, N))
    f.matmul(dx.arg(), arg, dout.arg(), m, N, K, transpose_b=not layout, b_scales=dev_s.arg() if dev_s else None)
    got = dout.download().astype(np.float64)
    want = x.astype(np.float64) @ full.astype(np.float64).T
    rest = np.arange(N) != 1
    assert np.all(got[:, 1] == np.inf), got[:, 1]
    # two f16 units of the result and the rounding of the weights that f16(weight * scale) has where it is used
    bar = 2.0 ** -9 * np.abs(want) + 2.0 ** -11 * (x.astype(np.float64) @ np.abs(full.astype(np.float64)).T) + 1e-4
    assert np.all(np.abs(got - want)[:, rest] <= bar[:, rest])
    for b in [dx, dout, dev_w] + ([dev_s] if dev_s else []):
        b.free()


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K", [160, 1056, 2080, 4064])  # blocks that do not fill the last wave's share, of one, two and four units
def test_one_input_row_infinite_last_block(K, weights, layout):
    announce("one input row, infinite last block", K, weights, layout)
    infinite_last_block(K, 24, 1, weights, layout)


@pytest.mark.parametrize("K", [96, 896, 4096])
def test_one_input_row_subnormal_weights(K):
    """F16 weights and inputs below the smallest normal number count with their values (exact in f32: products of two 11-bit numbers;
    the bar is the f16 rounding of the result and K f32 additions)."""
    announce("one input row, subnormal weights", K)
    f = ctx()
    rng = np.random.default_rng(K)
    N = 40
    w = (rng.integers(-1023, 1024, (N, K)) * 2.0 ** -24).astype(np.float16)  # subnormal
    x = rng.uniform(-200, 200, (1, K)).astype(np.float16)
    w[N // 2:] = rng.uniform(-1, 1, (N - N // 2, K)).astype(np.float16)  # (sums below the largest f16)
    x[0, ::3] = (rng.integers(-1023, 1024, len(x[0, ::3])) * 2.0 ** -24).astype(np.float16)
    for xv in (x, (rng.integers(-1023, 1024, (1, K)) * 2.0 ** -24).astype(np.float16)):
        dx, dw, dout = f.array(xv), f.array(orc.to_canonical(w)), f.zeros((1, N))
        f.matmul(dx.arg(), dw.arg(), dout.arg(), 1, N, K, transpose_b=False)
        xd, wd = xv.astype(np.float64), w.astype(np.float64)
        want, size = (xd @ wd.T)[0], (np.abs(xd) @ np.abs(wd).T)[0]
        err = np.abs(dout.download()[0].astype(np.float64) - want)
        assert np.all(err <= np.maximum(np.abs(want) * 2.0 ** -11, 2.0 ** -25) + K * 2.0 ** -24 * size)
        for b in (dx, dw, dout):
            b.free()
