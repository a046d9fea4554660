"""GPU parity of the one-launch kernel for chunks of input rows (FusedQkv and MatMul, fa_panel.h) where its split of the work
ends: row lengths around its 512-feature pieces, an odd number of feature blocks, weight rows that do not fill a tile or straddle
the matrices, one and several passes, passes spread over workgroups, the block-quantised arithmetic on either side of 12 rows.
Against the oracle with the bars of test_gpu_qkv.py."""
import numpy as np
import pytest

import foundry_attn as fa
import orc
from gpu_util import announce, ctx
from test_gpu_gemv_row import infinite_last_block
from test_gpu_qkv import _close, _data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K,N,NK,m,layout", [
    (32, 8, 8, 2, 1),          # one block
    (96, 40, 24, 11, 0),       # an odd number of blocks; the last row count of the weight stream's arithmetic
    (1024, 200, 40, 12, 1),    # the longest rows of the two-piece form, the first row count of the GEMM's arithmetic
    (1056, 72, 8, 16, 1),      # 33 blocks: just past it, 16 rows exactly
    (896, 264, 72, 33, 0),     # two passes, the second of one row
    (896, 64, 32, 100, 1),     # passes spread over workgroups
    (2048, 40, 16, 17, 0),
    (2080, 40, 16, 47, 1),     # 65 blocks: 16 rows per pass
    (3072, 24, 8, 5, 0),       # the longest rows it takes
    (3072, 4136, 1024, 20, 1), # as many weight rows per compute unit as two tiles hold, two passes
])
def test_chunk_in_one_launch(K, N, NK, m, layout, weights):
    announce("panel", K, N, NK, m, layout, weights)
    f = ctx()
    rng = np.random.default_rng(K + N + m)
    x, g, ws, bs = _data(rng, K, N, NK, m)
    res = rng.uniform(-1, 1, (m, N)).astype(np.float16)
    dx, dg, db, dres, dout = f.array(x), f.array(g), [f.array(b) for b in bs], f.array(res), f.zeros((m, N))
    outs = [f.zeros((m, n)) for n in (N, NK, NK)]
    scales, dev_s = None, []
    if weights == "f16":
        dev_w = [f.array(orc.to_canonical(w) if layout else w.reshape(-1)) for w in ws]
        arg = [w.arg() for w in dev_w]
        full = ws
    else:
        quant = [orc.quantize_q8_0(w) if weights == "q8" else orc.quantize_q4_0(w) for w in ws]
        dev_s = [f.array(s) for _, s in quant]
        scales = [s.arg() for s in dev_s]
        flat = [orc.to_canonical(q) if layout else q.reshape(-1) for q, _ in quant]
        dev_w = [f.array(q if weights == "q8" else orc.pack_q4_0(q)) for q in flat]
        arg = [w.arg() if weights == "q8" else w.arg((n, K), dtype=fa.DTYPE_Q4_0) for w, n in zip(dev_w, (N, NK, NK))]
        full = [orc.dequantize_blocks(q, s) for q, s in quant]
    if weights != "f16" and m < 12:
        want = orc.fused_qkv_q8(x, [q for q, _ in quant], [s for _, s in quant], gamma=g, biases=bs)
        want_mm = orc.matmul_gemv_q8(x, quant[0][0], quant[0][1], bs[0], res, 0, 32, 0.5, 0.75)
    else:
        want = orc.fused_qkv(x, *full, gamma=g, biases=bs, layout=0)
        want_mm = orc.matmul_gemv(x, full[0], bs[0], res, 0, 32, 0.5, 0.75)
    f.profile_reset()
    f.profile_enable(True)
    try:
        f.fused_qkv(dx.arg(), *arg, *[o.arg() for o in outs], K, N, NK, m, gamma=dg.arg(), biases=[b.arg() for b in db],
                    layout=layout, scales=scales)
        f.matmul(dx.arg(), arg[0], dout.arg(), m, N, K, bias=db[0].arg(), c=dres.arg(), transpose_b=not layout, alpha=0.5,
                 beta=0.75, b_scales=scales[0] if scales else None)
        f.synchronize()
        assert f.profile_query("fused_qkv_rows32_kernel")[0] == 1 and f.profile_query("matmul_rows32_kernel")[0] == 1
    finally:
        f.profile_enable(False)
    for o, w, name in zip(outs, want, "qkv"):
        got = o.download()
        assert np.all(np.isfinite(got)), name
        assert _close(got, w, K), (name, float(np.max(np.abs(got.astype(np.float64) - w.astype(np.float64)))))
    got, w = dout.download().astype(np.float64), want_mm.astype(np.float64)
    assert np.all(np.abs(got - w) <= 2 * np.maximum(np.abs(w), 2.0 ** -10) * 2.0 ** -10 + 1e-4), float(np.max(np.abs(got - w)))
    for b in [dx, dg, dres, dout] + db + outs + dev_w + dev_s:
        b.free()


@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K,N,NK,m,layout", [
    (2112, 4112, 520, 17, 0),   # 42 weight rows to a workgroup: three tiles, the last of 10 rows; the second pass of one row
    (3072, 4104, 512, 32, 1),   # the same, passes of 16 rows
    (3072, 4496, 1800, 18, 1),  # four tiles
    (2592, 3080, 520, 33, 0),   # three passes, an odd number of feature blocks
    (3072, 2056, 520, 64, 1),   # four passes, workgroups of the last group of eight without rows
])
def test_long_rows_a_workgroup_for_each_pass(K, N, NK, m, layout, weights):
    test_chunk_in_one_launch(K, N, NK, m, layout, weights)


@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K,N,NK,m,layout", [
    (2048, 2056, 256, 40, 1),  # 34 weight rows to a workgroup: two rows in a third tile; three passes, the last of 8 rows
    (2048, 2304, 384, 64, 0),  # three full tiles, four passes
    (1056, 3000, 544, 17, 1),  # two tiles, a pass of one row
    (640, 1504, 272, 33, 0),   # two tiles of short rows
    (896, 1024, 128, 41, 1),   # one tile
])
def test_shorter_rows_a_workgroup_for_each_pass(K, N, NK, m, layout, weights):
    test_chunk_in_one_launch(K, N, NK, m, layout, weights)


@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K,N,NK,m,layout", [
    (96, 776, 40, 9, 1),       # 8 input rows to a workgroup: a second pass of one row; the weight stream's arithmetic of block-quantised weights
    (896, 896, 128, 16, 0),    # two full passes
    (2048, 1800, 120, 11, 1),  # longer rows, 16 weight rows to a workgroup
    (2048, 2048, 264, 17, 0),  # three passes of two tiles with the norm, two of 16 rows without
    (1056, 1000, 136, 23, 1),  # three, the last of 7 rows
    (640, 1200, 40, 90, 1),    # six passes of 16
])
def test_passes_of_8_rows(K, N, NK, m, layout, weights):
    test_chunk_in_one_launch(K, N, NK, m, layout, weights)


def test_long_rows_in_five_tiles():
    test_chunk_in_one_launch(2592, 3840, 640, 64, 1, "f16")  # 80 weight rows to a workgroup, block-quantised as a GEMM


@pytest.mark.parametrize("K,N,NK,m,layout,weights", [
    (2592, 4104, 520, 40, 0, "f16"),  # three passes by one workgroup with two tiles (the product without a norm: 18 weight rows)
    (2592, 3000, 24, 40, 0, "f16"),   # the product in one tile
    (2592, 4104, 520, 40, 0, "q8"),
    (2592, 4104, 520, 33, 1, "q8"),   # the last pass of one row
    (2592, 4104, 520, 33, 1, "q4"),
    (2592, 1160, 64, 35, 0, "q8"),    # one tile, a workgroup for each pass
    (2592, 264, 72, 20, 1, "q4"),
])
def test_long_rows_walked_over(K, N, NK, m, layout, weights):
    """Rows of more than 2048 features whose workgroups keep all their weights and go on to further passes (which of them do:
    test_panel_plan.py)."""
    test_chunk_in_one_launch(K, N, NK, m, layout, weights)


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K,m", [(32, 2), (96, 11), (96, 12), (896, 33), (1056, 5), (2016, 20), (2080, 5), (2080, 17)])
def test_chunk_in_one_launch_infinite_last_block(K, m, weights, layout):
    """Row lengths of every number of feature pieces whose blocks do not fill a wave's share, odd and even in number."""
    announce("panel, infinite last block", K, m, weights, layout)
    infinite_last_block(K, 40, m, weights, layout)


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("K,N,NK,m", [(1024, 40, 24, 3), (1056, 40, 24, 2), (1088, 72, 8, 11), (1120, 200, 40, 7), (1152, 40, 24, 4), (2048, 264, 72, 11), (2080, 40, 24, 2),
                                      (3040, 40, 16, 11), (3072, 4136, 1024, 6)])
def test_q4_weights_turned_into_operand_order(K, N, NK, m, layout):
    """Q4_0 with per-block sums (2 to 11 rows): the weights of four blocks go through LDS from the longest rows that do not, with one,
    two, three and four blocks in a row's last request, one and two tiles of weight rows, both layouts."""
    test_chunk_in_one_launch(K, N, NK, m, layout, "q4")


@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K,N,NK,m", [(96, 40, 24, 8), (96, 40, 24, 9), (1056, 72, 8, 8), (1056, 72, 8, 24), (2080, 40, 24, 8), (2080, 40, 24, 9), (2080, 264, 72, 24),
                                      (2048, 72, 8, 25), (2080, 40, 16, 25), (896, 64, 32, 40), (896, 64, 32, 73), (3072, 4136, 1024, 8)])
def test_rows_absent_from_a_pass(K, N, NK, m, weights):
    """A wave's rows of a pass are asked for and normalised only where they are there, and there is a form for a single row per wave:
    one row group less than a pass holds and one row more, in a first, a second and a last pass, rows of two, four and six pieces."""
    test_chunk_in_one_launch(K, N, NK, m, 1, weights)


@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K,H,Hkv,D,m", [
    (96, 6, 1, 64, 3),        # a pair of rows per workgroup
    (1024, 14, 2, 64, 20),    # three
    (96, 14, 2, 64, 100),     # eight, several passes
    (2048, 16, 2, 128, 8),    # five
    (2080, 16, 2, 128, 33),   # eight: passes spread over workgroups
    (96, 28, 2, 128, 17),     # the most that one tile holds
    (96, 30, 2, 128, 9),      # past it: two tiles
    (3072, 24, 8, 128, 32),   # 20 pairs: 16 in two tiles, 4 in a third
    (2816, 24, 12, 128, 19),  # 24: the third is full
    (3072, 24, 8, 128, 40),   # 32 in four tiles
    (2048, 16, 4, 128, 40),   # 20 of shorter rows
    (1024, 14, 2, 64, 60),    # 9 in two tiles, four passes
    (896, 14, 2, 64, 13),     # 5, passes of 8 rows
    (2048, 16, 2, 128, 24),   # 16 in two tiles, passes of 8 rows
])
def test_neox_pairs_in_one_tile(K, H, Hkv, D, m, weights, layout=1, norm=True):
    """Up to 16 weight rows per workgroup, and in the last of an odd number of tiles, both halves of NeoX pairs lie in one tile: the fused
    write stage equals the two ops to the bit, in both pairings."""
    announce("neox pairs in one tile", K, H, Hkv, D, m, weights, layout, norm)
    f = ctx()
    rng = np.random.default_rng(K + H + m)
    N, NK = H * D, Hkv * D
    x, g, ws, bs = _data(rng, K, N, NK, m)
    scales, dev_s = None, []
    if weights == "f16":
        dev_w = [f.array(orc.to_canonical(w) if layout else w.reshape(-1)) for w in ws]
        arg = [w.arg() for w in dev_w]
    else:
        quant = [orc.quantize_q8_0(w) if weights == "q8" else orc.quantize_q4_0(w) for w in ws]
        dev_s = [f.array(s) for _, s in quant]
        scales = [s.arg() for s in dev_s]
        flat = [orc.to_canonical(q) if layout else q.reshape(-1) for q, _ in quant]
        dev_w = [f.array(q if weights == "q8" else orc.pack_q4_0(q)) for q in flat]
        arg = [w.arg() if weights == "q8" else w.arg((n, K), dtype=fa.DTYPE_Q4_0) for w, n in zip(dev_w, (N, NK, NK))]
    dx, dg, db = f.array(x), f.array(g), [f.array(b) for b in bs]
    outs = [f.zeros((m, n)) for n in (N, NK, NK)]
    cos, sin = fa.rope_tables(5e5, D, m + 3)
    dcos, dsin = f.array(cos), f.array(sin)
    rot = [[f.zeros((H, m, D)), f.zeros((Hkv, m + 3, D)), f.zeros((Hkv, m + 3, D))] for _ in range(2)]
    kw = dict(gamma=dg.arg() if norm else None, biases=[b.arg() for b in db], layout=layout, scales=scales)
    f.fused_qkv(dx.arg(), *arg, *[o.arg() for o in outs], K, N, NK, m, **kw)
    for mode in (fa.ROPE_NEOX, fa.ROPE_NORMAL):
        p = fa.KvPrepFusedParams.make(H, Hkv, D, m, 2, m + 3, mode)
        f.kv_prep_fused(*[o.arg() for o in outs], *[t.arg() for t in rot[0]], dcos.arg(), dsin.arg(), p)
        f.profile_reset()
        f.profile_enable(True)
        try:
            f.fused_qkv_kv_prep(dx.arg(), *arg, K, rot[1][0].arg(), dcos.arg(), dsin.arg(), p, k_cache=rot[1][1].arg(), v_cache=rot[1][2].arg(), **kw)
            f.synchronize()
            assert f.profile_query("fused_qkv_rows32_rope_kernel")[0] == 1
        finally:
            f.profile_enable(False)
        for one, two in zip(rot[0], rot[1]):
            got, want = two.download(), one.download()
            assert np.any(want) and np.array_equal(got.view(np.uint16), want.view(np.uint16)), mode
    for b in [dx, dg, dcos, dsin] + db + outs + dev_w + dev_s + rot[0] + rot[1]:
        b.free()


@pytest.mark.parametrize("K,H,Hkv,D,m", [(3072, 24, 8, 128, 64), (2592, 36, 1, 128, 57)])
def test_neox_pairs_in_five_tiles(K, H, Hkv, D, m):
    """40 pairs to a workgroup, 32 in two pairs of tiles and 8 in a fifth; 38 of them, and a last pass of 9 rows."""
    test_neox_pairs_in_one_tile(K, H, Hkv, D, m, "f16")


@pytest.mark.parametrize("K,H,Hkv,D,m,weights,layout,norm", [
    (2592, 40, 1, 128, 33, "f16", 0, True),  # two tiles, three passes by one workgroup
    (2592, 24, 3, 128, 40, "f16", 0, False),  # one tile
    (2592, 40, 1, 128, 33, "q8", 1, True),
    (2592, 19, 1, 64, 35, "q8", 1, True),    # one tile, a workgroup for each pass
    (2592, 40, 1, 128, 33, "q4", 0, True),
    (2592, 19, 1, 64, 35, "q4", 1, True),
])
def test_rotation_of_long_rows_walked_over(K, H, Hkv, D, m, weights, layout, norm):
    test_neox_pairs_in_one_tile(K, H, Hkv, D, m, weights, layout, norm)


@pytest.mark.parametrize("weights", ["q8", "q4"])
def test_sums_of_long_rows_are_as_exact_as_the_tiles(weights):
    """The f32 sums behind the rounding to f16, from 2^10 (sum - its f16 value), against 64 bits: the error of 56 rows of 3072 features is no
    larger than that of the GEMM's tiles, which take more rows than that."""
    K, N, m, S = 3072, 2048, 56, 2.0 ** 10
    announce("panel, error of the sums", weights)
    f = ctx()
    rng = np.random.default_rng(5)
    x = rng.normal(size=(m, K)).astype(np.float16)
    w = (rng.normal(size=(N, K)) * K ** -0.5).astype(np.float16)
    q, s = orc.quantize_q8_0(w) if weights == "q8" else orc.quantize_q4_0(w)
    exact = x.astype(np.float64) @ orc.dequantize_blocks(q, s).astype(np.float64).T
    c = exact.astype(np.float16)
    dw = f.array(q.reshape(-1) if weights == "q8" else orc.pack_q4_0(q.reshape(-1)))
    arg = dw.arg() if weights == "q8" else dw.arg((N, K), dtype=fa.DTYPE_Q4_0)
    dx, ds, dc, do, error = f.array(x), f.array(s), f.array(c), f.zeros((m, N)), []
    for min_m, name in ((0, "matmul_rows32_kernel"), (1, "matmul_gemm_kernel")):
        f.set_gemm_min_m(min_m)
        f.profile_reset()
        f.profile_enable(True)
        try:
            f.matmul(dx.arg(), arg, do.arg(), m, N, K, c=dc.arg(), transpose_b=True, alpha=S, beta=-S, b_scales=ds.arg())
            f.synchronize()
            assert f.profile_query(name)[0] == 1
        finally:
            f.profile_enable(False)
            f.set_gemm_min_m()
        error.append(np.sqrt(np.mean((do.download() / S - (exact - c)) ** 2) / np.mean(exact ** 2)) * 2.0 ** 24)
    assert 0 < error[0] <= error[1] < 4, error
    for b in (dx, dw, ds, dc, do):
        b.free()
