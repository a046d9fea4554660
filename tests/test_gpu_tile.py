"""GPU parity of the tile kernels of FusedQkv and MatMul (fa_tile.h): fewer steps than stages, steps that do not fill the unrolled
loop, tiles cut off by the last input or weight row, every tile shape (by the number of tiles that the launch has), tiles that hold
rows of two matrices, and both head widths of the NeoX write stage. Against the oracle with the bars of test_gpu_qkv.py; the fused
write stage against the two ops, bit for bit."""
import numpy as np
import pytest

import foundry_attn as fa
import orc
from gpu_util import announce, bits, ctx
from test_gpu_paged import Paged
from test_gpu_qkv import _close, _data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K,H,Hkv,D,m,layout", [
    (64, 3, 1, 64, 12, 1),        # one step, one ragged tile
    (192, 1, 1, 128, 65, 0),      # three steps, a second tile of one row
    (320, 5, 1, 64, 130, 1),      # five steps
    (896, 2, 1, 64, 513, 0),      # fourteen steps: seven pairs, scales of three and a half units
    (128, 16, 2, 64, 1030, 1),    # 128 x 64 tiles
    (576, 14, 2, 64, 2047, 0),    # 128 x 128 tiles
    (128, 40, 8, 64, 1000, 1),    # 256 x 128 tiles
    (320, 40, 8, 64, 1000, 0),
    (192, 32, 4, 64, 520, 1),     # 64 x 96 tiles, both ops; the last one a third full, K and V of two thirds of one
    (192, 32, 4, 64, 520, 0),
    (1088, 16, 2, 128, 577, 1),   # and Q4_0 with steps of each wave's own, seventeen of them
    (1024, 16, 2, 128, 524, 0),
    (128, 24, 8, 128, 2040, 1),   # F16: 256 x 160 tiles, some with rows of two matrices
    (192, 24, 8, 128, 2048, 0),
])
def test_tiles(K, H, Hkv, D, m, layout, weights):
    announce("tiles", K, H, Hkv, D, m, layout, weights)
    f = ctx()
    rng = np.random.default_rng(K + H + m)
    N, NK = H * D, Hkv * D
    x, g, ws, bs = _data(rng, K, N, NK, m)
    res = rng.uniform(-1, 1, (m, N)).astype(np.float16)
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
    dx, dg, db, dres, dout = f.array(x), f.array(g), [f.array(b) for b in bs], f.array(res), f.zeros((m, N))
    outs = [f.zeros((m, n)) for n in (N, NK, NK)]
    cos, sin = fa.rope_tables(5e5, D, m + 3)
    dcos, dsin = f.array(cos), f.array(sin)
    rot = [[f.zeros((H, m, D)), f.zeros((Hkv, m + 3, D)), f.zeros((Hkv, m + 3, D))] for _ in range(2)]
    kw = dict(gamma=dg.arg(), biases=[b.arg() for b in db], layout=layout, scales=scales)
    try:
        f.set_gemm_min_m(12)
        f.fused_qkv(dx.arg(), *arg, *[o.arg() for o in outs], K, N, NK, m, **kw)
        for o, w, name in zip(outs, orc.fused_qkv(x, *full, gamma=g, biases=bs, layout=0), "qkv"):
            assert _close(o.download(), w, K), name
        for mode in (fa.ROPE_NEOX, fa.ROPE_NORMAL):
            p = fa.KvPrepFusedParams.make(H, Hkv, D, m, 2, m + 3, mode)
            f.kv_prep_fused(*[o.arg() for o in outs], *[t.arg() for t in rot[0]], dcos.arg(), dsin.arg(), p)
            f.fused_qkv_kv_prep(dx.arg(), *arg, K, rot[1][0].arg(), dcos.arg(), dsin.arg(), p, k_cache=rot[1][1].arg(),
                                v_cache=rot[1][2].arg(), **kw)
            for one, two in zip(rot[0], rot[1]):
                assert np.array_equal(bits(one.download()), bits(two.download())), mode
        f.matmul(dx.arg(), arg[0], dout.arg(), m, N, K, bias=db[0].arg(), c=dres.arg(), transpose_b=layout == 0, alpha=0.5, beta=0.75,
                 b_scales=scales[0] if scales else None)
        want = orc.matmul_gemv(x, full[0], bs[0], res, 0, 32, 0.5, 0.75).astype(np.float64)
        assert np.all(np.abs(dout.download() - want) <= 2 * np.maximum(np.abs(want), 2.0 ** -10) * 2.0 ** -10 + 1e-4)
    finally:
        f.set_gemm_min_m()
    for b in dev_w + dev_s + [dx, dg, dres, dout, dcos, dsin] + db + outs + rot[0] + rot[1]:
        b.free()


@pytest.mark.parametrize("K,N,m", [(256, 200, 130), (1024, 520, 577), (192, 2056, 520)])  # 64 x 64 tiles, with steps of each wave's own, 64 x 96
@pytest.mark.parametrize("weights", ["f16", "q8"])
def test_residual_asked_for_ahead_of_the_sums(K, N, m, weights):
    """Every tile reads its own places of the residual, whatever is done with the ones past the last row: in place of it, the output is the same bits."""
    announce("residual ahead", K, N, m, weights)
    f = ctx()
    rng = np.random.default_rng(K + N + m)
    x, w = rng.uniform(-1, 1, (m, K)).astype(np.float16), (rng.uniform(-1, 1, (N, K)) / 16).astype(np.float16)
    res = rng.uniform(-1, 1, (m, N)).astype(np.float16)
    q, s = orc.quantize_q8_0(w)
    dx, dres, dout = f.array(x), f.array(res), f.zeros((m, N))
    dw, ds = f.array(q if weights == "q8" else w), f.array(s)
    kw = dict(transpose_b=True, beta=0.75, b_scales=ds.arg() if weights == "q8" else None)
    try:
        f.set_gemm_min_m(12)
        f.matmul(dx.arg(), dw.arg(), dout.arg(), m, N, K, c=dres.arg(), **kw)
        got = dout.download()
        f.matmul(dx.arg(), dw.arg(), dres.arg(), m, N, K, c=dres.arg(), **kw)
        assert np.array_equal(bits(dres.download()), bits(got))
    finally:
        f.set_gemm_min_m()
    for b in (dx, dres, dout, dw, ds):
        b.free()
    full = orc.dequantize_blocks(q, s) if weights == "q8" else w
    want = orc.matmul_gemv(x, full, None, res, 0, 32, 1.0, 0.75).astype(np.float64)
    assert np.all(np.abs(got - want) <= 2 * np.maximum(np.abs(want), 2.0 ** -10) * 2.0 ** -10 + 1e-4)  # (as test_tiles)


@pytest.mark.parametrize("row_tiles", [1, 8, 9, 11, 33])  # weight tiles of all input tiles in a row, and in fours, the last ones of one to four
@pytest.mark.parametrize("col_tiles", [1, 2, 3, 4, 5, 6, 7])
def test_every_output_tile_once(row_tiles, col_tiles):
    """64 x 64 tiles (64 features: a launch of one step) of whole numbers, whose sums f16 holds: exact, in every tile of the launch."""
    announce("every tile", row_tiles, col_tiles)
    f = ctx()
    K, m, N = 64, 64 * row_tiles - 3, 64 * col_tiles - 8
    rng = np.random.default_rng(row_tiles * 8 + col_tiles)
    x, w = rng.integers(-3, 4, (m, K)).astype(np.float16), rng.integers(-3, 4, (N, K)).astype(np.float16)
    dx, dw, dout = f.array(x), f.array(w), f.array(np.full((m, N), np.nan, np.float16))
    try:
        f.set_gemm_min_m(12)
        f.set_gemm_variant(3)
        f.matmul(dx.arg(), dw.arg(), dout.arg(), m, N, K, transpose_b=True)
    finally:
        f.set_gemm_variant()
        f.set_gemm_min_m()
    assert np.array_equal(dout.download(), (x.astype(np.float32) @ w.astype(np.float32).T).astype(np.float16))
    for b in (dx, dw, dout):
        b.free()


@pytest.mark.parametrize("weights", ["q8", "q4"])
@pytest.mark.parametrize("K,H,Hkv,D,m,layout", [
    (960, 2, 1, 64, 65, 1),       # the last length whose steps the waves of a tile share
    (1024, 2, 1, 64, 65, 1),      # four steps for each wave, a second tile of one row
    (1088, 1, 1, 128, 64, 0),     # a step more for one wave
    (1152, 3, 1, 64, 130, 1),     # for two of four; scales of four and a half units
    (1216, 5, 1, 64, 12, 0),      # for three, a ragged tile
    (2112, 2, 2, 128, 33, 1),
    (4096, 1, 1, 64, 70, 0),      # all of a compute unit's LDS
    (4096, 1, 1, 128, 20, 1),
    (4160, 1, 1, 64, 20, 1),      # past it
])
def test_tiles_with_steps_of_each_waves_own(K, H, Hkv, D, m, layout, weights):
    """Block-quantised 64 x 64 tiles: every wave has every fourth step of 64 features from 1024 to 4096 of them."""
    ctx().set_gemm_variant(3)
    try:
        test_tiles(K, H, Hkv, D, m, layout, weights)
    finally:
        ctx().set_gemm_variant()


@pytest.mark.parametrize("weights", ["q8", "q4"])
@pytest.mark.parametrize("K,H,Hkv,D,m,layout", [
    (64, 3, 1, 64, 12, 1),        # one step, fewer than stages
    (448, 2, 1, 64, 65, 0),       # seven: the unrolled loop is cut off; scales of one unit and three quarters
    (576, 1, 1, 128, 64, 1),      # nine steps
    (896, 14, 2, 64, 448, 1),     # 252 tiles
    (896, 14, 2, 64, 449, 0),     # 288: tiles of 64 x 64 again
    (1088, 1, 1, 128, 130, 1),
    (2112, 2, 2, 64, 33, 0),
    (8256, 1, 1, 64, 70, 1),      # past the features that the 64 x 64 forms with more stages have room for
])
def test_tiles_of_32_weight_rows(K, H, Hkv, D, m, layout, weights):
    test_tiles(K, H, Hkv, D, m, layout, weights)


@pytest.mark.parametrize("weights", ["q8", "q4"])
@pytest.mark.parametrize("K,H,Hkv,D,m,layout", [
    (192, 1, 1, 128, 65, 0), (896, 2, 1, 64, 513, 0), (1024, 2, 1, 64, 65, 1), (1088, 1, 1, 128, 64, 0), (1216, 5, 1, 64, 12, 0),
    (4096, 1, 1, 64, 70, 0), (4160, 1, 1, 64, 20, 1)])
def test_tiles_of_64_weight_rows_by_name(K, H, Hkv, D, m, layout, weights):
    """The 64 x 64 forms at sizes that the narrower tiles take of themselves."""
    f = ctx()
    f.set_gemm_variant(3)
    try:
        test_tiles(K, H, Hkv, D, m, layout, weights)
    finally:
        f.set_gemm_variant()


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("order", ["qkv", "kvq", "vqk"])
def test_weights_anywhere_in_memory(order, layout):
    """F16 tiles that hold rows of two matrices: the kernel, and so the bits, of a launch do not depend on where the matrices lie. The
    bar is two f16 units of the result and six roots of 2 n roundings (test_f16_sums_are_added_in_parts) of a chain of 64 products."""
    announce("weights anywhere", order, layout)
    f = ctx()
    K, N, NK, m = 1024, 3072, 1024, 2040
    rng = np.random.default_rng(K + m + layout)
    x = rng.normal(size=(m, K)).astype(np.float16)
    ws = [(rng.normal(size=(n, K)) * K ** -0.5).astype(np.float16) for n in (N, NK, NK)]
    flat = [orc.to_canonical(w) if layout else w.reshape(-1) for w in ws]
    far = (1 << 32) + (1 << 20)
    pool = f.empty((2 * far + N * K * 2,), np.uint8)
    dx, outs = f.array(x), [f.zeros((m, n)) for n in (N, NK, NK)]
    got = []
    for apart in (False, True):
        at, end = [0, 0, 0], 0
        for i in ("qkv".index(c) for c in order):
            at[i], end = end, end + (far if apart else flat[i].nbytes)
        args = []
        for w, o in zip(flat, at):
            fa.check(f.lib.fa_upload(f.h, pool.ptr, o, w.ctypes.data, w.nbytes))
            args.append(pool.arg(w.shape, offset=o, dtype=fa.DTYPE_F16))
        f.fused_qkv(dx.arg(), *args, *[o.arg() for o in outs], K, N, NK, m, layout=layout)
        got.append([o.download() for o in outs])
    for near, apart, w in zip(*got, ws):
        assert np.array_equal(bits(near), bits(apart))
        want = x.astype(np.float64) @ w.astype(np.float64).T
        assert np.all(np.abs(near - want) <= 2.0 ** -9 * np.abs(want) + 6 * 0.42 * 8 * 2.0 ** -24 * np.sqrt(np.mean(want ** 2)) + 2.0 ** -23)
    for b in [pool, dx] + outs:
        b.free()


@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K,N,NK,m,panel,finish", [
    (2048, 8192, 1024, 16, True, False),    # one round of workgroups: the panel up to 32 rows
    (2048, 8192, 1024, 48, False, False),   # many weight rows: its passes cost more than the norm's launch and the tiles
    (2048, 2048, 256, 64, True, False),
    (1024, 4096, 1024, 40, "f16", False),   # no side a tenth ahead (block-quantised: more than one pass per compute unit)
    (1024, 4096, 1024, 100, False, False),
    (896, 896, 128, 400, "f16", False),
    (896, 896, 128, 417, False, False),
    (3072, 40, 24, 48, True, False),        # a few weight rows
    (4096, 512, 128, 16, False, None),      # about the line between whole and divided
    (8192, 512, 64, 12, False, True),       # few tiles over many features: divided
    (8192, 512, 64, 130, False, True),
    (3200, 8192, 512, 12, False, False),    # enough tiles
    (16384, 256, 64, 20, False, True),
])
def test_route_of_a_chunk(K, N, NK, m, panel, finish, weights):
    """Which launches a chunk takes is decided by what they are estimated to take; whichever it is, the outputs hold to the oracle.
    (The longest rows without the norm: its f16 roundings differ from the oracle's in isolated elements, 60 in a million, more of
    them in a row of 8192 than the bar allows for, whatever kernel multiplies them.)"""
    announce("route of a chunk", K, N, NK, m, weights)
    panel = panel is True or panel == weights
    f = ctx()
    rng = np.random.default_rng(K + N + m)
    x, g, ws, bs = _data(rng, K, N, NK, m)
    norm = K <= 4096
    scales, dev_s = None, []
    if weights == "f16":
        dev_w = [f.array(orc.to_canonical(w)) for w in ws]
        arg, full = [w.arg() for w in dev_w], ws
    else:
        quant = [orc.quantize_q8_0(w) if weights == "q8" else orc.quantize_q4_0(w) for w in ws]
        dev_s = [f.array(s) for _, s in quant]
        scales = [s.arg() for s in dev_s]
        flat = [orc.to_canonical(q) for q, _ in quant]
        dev_w = [f.array(q if weights == "q8" else orc.pack_q4_0(q)) for q in flat]
        arg = [w.arg() if weights == "q8" else w.arg((n, K), dtype=fa.DTYPE_Q4_0) for w, n in zip(dev_w, (N, NK, NK))]
        full = [orc.dequantize_blocks(q, s) for q, s in quant]
    dx, dg, db = f.array(x), f.array(g), [f.array(b) for b in bs]
    outs = [f.zeros((m, n)) for n in (N, NK, NK)]
    f.profile_reset()
    f.profile_enable(True)
    try:
        f.fused_qkv(dx.arg(), *arg, *[o.arg() for o in outs], K, N, NK, m, gamma=dg.arg() if norm else None,
                    biases=[b.arg() for b in db], layout=1, scales=scales)
        f.synchronize()
        assert f.profile_query("fused_qkv_rows32_kernel")[0] == int(panel) and f.profile_query("fused_qkv_gemm_kernel")[0] == int(not panel)
        if finish is not None:
            assert f.profile_query("gemm_finish_kernel")[0] == int(finish)
    finally:
        f.profile_enable(False)
    for o, w, name in zip(outs, orc.fused_qkv(x, *full, gamma=g if norm else None, biases=bs, layout=0), "qkv"):
        assert _close(o.download(), w, K), name
    for b in dev_w + dev_s + [dx, dg] + db + outs:
        b.free()


def _quantised(f, rng, K, N, m, weights):
    x = rng.uniform(-1, 1, (m, K)).astype(np.float16)
    q, s = (orc.quantize_q8_0 if weights == "q8" else orc.quantize_q4_0)(rng.uniform(-0.1, 0.1, (N, K)).astype(np.float16))
    flat = orc.to_canonical(q)
    dev_w = f.array(flat if weights == "q8" else orc.pack_q4_0(flat))
    return x, orc.dequantize_blocks(q, s), s, dev_w, dev_w.arg() if weights == "q8" else dev_w.arg((N, K), dtype=fa.DTYPE_Q4_0)


@pytest.mark.parametrize("weights", ["q8", "q4"])
@pytest.mark.parametrize("K,N,NK,m,panel", [
    (640, 896, 192, 192, True), (640, 896, 192, 193, False),     # 240, 280 pieces of 32 x 32 rows
    (896, 960, 32, 256, True), (896, 960, 32, 257, False),       # 256, 288
    (960, 1856, 64, 256, False), (960, 1856, 64, 128, True),     # 496, 248
    (1280, 1984, 64, 124, False),                                # 264
])
def test_route_of_a_quantised_chunk_with_a_norm(K, N, NK, m, panel, weights):
    test_route_of_a_chunk(K, N, NK, m, panel, None, weights)


@pytest.mark.parametrize("weights", ["q8", "q4"])
@pytest.mark.parametrize("K,N,m,panel", [
    (896, 896, 193, True), (896, 896, 288, True),   # up to a pass for each compute unit
    (896, 896, 289, False),
    (1024, 512, 512, True), (1024, 512, 513, False),  # the most input rows
    (1056, 256, 193, False),                          # longer rows
])
def test_route_of_a_product_of_many_rows(K, N, m, panel, weights):
    """Block-quantised weights without a norm: the panel kernel while the passes fit one round of workgroups."""
    announce("route of a product", K, N, m, weights)
    f = ctx()
    rng = np.random.default_rng(K + N + m)
    x, full, s, dev_w, arg = _quantised(f, rng, K, N, m, weights)
    res = rng.uniform(-1, 1, (m, N)).astype(np.float16)
    dx, ds, dres, dout = f.array(x), f.array(s), f.array(res), f.zeros((m, N))
    f.profile_reset()
    f.profile_enable(True)
    try:
        f.matmul(dx.arg(), arg, dout.arg(), m, N, K, c=dres.arg(), transpose_b=False, beta=0.75, b_scales=ds.arg())
        f.synchronize()
        assert f.profile_query("matmul_rows32_kernel")[0] == int(panel) and f.profile_query("matmul_gemm_kernel")[0] == int(not panel)
    finally:
        f.profile_enable(False)
    want = orc.matmul_gemv(x, full, None, res, 0, 32, 1.0, 0.75).astype(np.float64)
    assert np.all(np.abs(dout.download() - want) <= 2 * np.maximum(np.abs(want), 2.0 ** -10) * 2.0 ** -10 + 1e-4)
    for b in (dx, ds, dres, dout, dev_w):
        b.free()


@pytest.mark.parametrize("weights", ["q8", "q4"])
@pytest.mark.parametrize("K,m", [
    (4096, 70), (4160, 70),    # the last row whose scales fit every tile's part of LDS, and the first past it: 64 x 64 tiles
    (8192, 70), (8256, 70),    # ... of eight small stages up to here
    (16384, 130),              # the longest row
    (16448, 70),               # past it: operand tiles through registers
])
def test_long_quantised_rows(K, m, weights):
    """Each kernel that takes such rows (operand tiles through registers, 128 x 128 tiles where the scales fit, 64 x 64, by choice)."""
    announce("long quantised rows", K, m, weights)
    f = ctx()
    N = 200
    x, full, s, dev_w, arg = _quantised(f, np.random.default_rng(K + m), K, N, m, weights)
    dx, ds, dout = f.array(x), f.array(s), f.zeros((m, N))
    got = []
    try:
        for variant in (0, 1, 2, 3):
            f.set_gemm_variant(variant)
            f.matmul(dx.arg(), arg, dout.arg(), m, N, K, transpose_b=False, b_scales=ds.arg())
            got.append(dout.download())
    finally:
        f.set_gemm_variant()
    want = orc.matmul_gemv(x, full, None, None, 0, 32, 1.0, 0.0).astype(np.float64)
    for g in got:
        assert np.all(np.abs(g - want) <= 2 * np.maximum(np.abs(want), 2.0 ** -10) * 2.0 ** -10 + 1e-4)
    for b in (dx, ds, dev_w, dout):
        b.free()


@pytest.mark.parametrize("weights", ["q8", "q4"])
@pytest.mark.parametrize("K,m", [(128, 1), (2048, 1), (64, 5), (896, 5), (896, 20), (3072, 40), (64, 500), (896, 500)])
def test_scales_at_any_half(K, m, weights):
    """Scales that begin at an odd f16: the kernels that read them in pairs leave them to others or read them one by one."""
    announce("scales at any half", K, m, weights)
    f = ctx()
    N = 72
    x, full, s, dev_w, arg = _quantised(f, np.random.default_rng(K + m), K, N, m, weights)
    dx, dout = f.array(x), f.zeros((m, N))
    moved = np.concatenate([np.full(1, 99.0, np.float16), s.reshape(-1), np.full(1, 99.0, np.float16)])
    ds = f.array(moved)
    f.matmul(dx.arg(), arg, dout.arg(), m, N, K, transpose_b=False, b_scales=ds.arg(s.shape, offset=2))
    want = x.astype(np.float64) @ full.astype(np.float64).T
    # two f16 units of the result and, from 12 rows on, the rounding of f16(weight * scale)
    bar = 2.0 ** -9 * np.abs(want) + 2.0 ** -11 * (np.abs(x.astype(np.float64)) @ np.abs(full.astype(np.float64)).T) + 1e-4
    assert np.all(np.abs(dout.download() - want) <= bar)
    for b in (dx, ds, dev_w, dout):
        b.free()


@pytest.mark.parametrize("K,m,variant,N", [(3072, 300, 0, 256), (3072, 300, 1, 256), (3072, 300, 2, 256), (2048, 1500, 0, 256), (3104, 300, 0, 256),
                                           (2048, 1300, 0, 3072), (1536, 1600, 0, 2560)])
def test_f16_sums_are_added_in_parts(K, m, variant, N):
    """The f32 sums of F16 weights behind the output's rounding: out = sums - f16(exact), so that what is left shows them to 2^-24.
    A chain of n matrix products of 16 features rounds 2 n times by 0.42 x 2^-24 rms of a partial sum that is half the final one in
    the mean square: 0.42 sqrt(n) x 2^-24 of the sums' size, 1.7 for parts of 256 features; adding N / 256 parts up rounds by
    0.42 sqrt(N / 512), 1.0 over 3072. Together 2.0, the bar 1.5 times that; one chain over 2048 features would be 4.7, over 3072
    5.8."""
    announce("F16 sums", K, m, variant, N)
    f = ctx()
    rng = np.random.default_rng(K + m)
    x = rng.normal(size=(m, K)).astype(np.float16)
    w = (rng.normal(size=(N, K)) * K ** -0.5).astype(np.float16)
    exact = x.astype(np.float64) @ w.astype(np.float64).T
    rounded = exact.astype(np.float16)
    dx, dw, dres, dout = f.array(x), f.array(w.reshape(-1)), f.array(-rounded), f.zeros((m, N))
    try:
        f.set_gemm_variant(variant)
        f.matmul(dx.arg(), dw.arg(), dout.arg(), m, N, K, c=dres.arg(), transpose_b=True, beta=1.0)
        err = dout.download().astype(np.float64) - (exact - rounded.astype(np.float64))
    finally:
        f.set_gemm_variant()
    assert np.sqrt(np.mean(err ** 2) / np.mean(exact ** 2)) * 2 ** 24 <= 3.0, np.sqrt(np.mean(err ** 2) / np.mean(exact ** 2)) * 2 ** 24
    for b in (dx, dw, dres, dout):
        b.free()


@pytest.mark.parametrize("K,m,N,chains", [
    (3072, 340, 3072, 4),  # 64 x 96 tiles
    (896, 200, 4864, 4),
    (4096, 288, 4096, 4),
    (2048, 200, 2048, 8),  # 64 x 64 with steps of each wave's own
    (1088, 400, 3072, 4),
])
def test_quantised_sums_are_several_chains(K, m, N, chains):
    """The f32 sums of Q8_0 weights whose scales are powers of two (their products with the weights are exact), as in
    test_f16_sums_are_added_in_parts: chains of n products of 16 features round by 0.42 sqrt(n) x 2^-24 of the sums' size, the output
    (f16 of a remainder of 2^-11 of them at most, uniform) by 0.7. With half as many chains the first is 1.41 times that."""
    announce("quantised sums", K, m, N, chains)
    f = ctx()
    rng = np.random.default_rng(K + m)
    x = rng.normal(size=(m, K)).astype(np.float16)
    q = np.clip(np.round(rng.normal(size=(N, K)) * 36), -127, 127).astype(np.int8)
    s = (2.0 ** rng.integers(-11, -9, size=(N, K // 32))).astype(np.float16)
    full = q.astype(np.float64) * np.repeat(s.astype(np.float64), 32, axis=1)
    exact = x.astype(np.float64) @ full.T
    rounded = exact.astype(np.float16)
    dx, dw, ds, dres, dout = f.array(x), f.array(q.reshape(-1)), f.array(s), f.array(-rounded), f.zeros((m, N))
    f.matmul(dx.arg(), dw.arg(), dout.arg(), m, N, K, c=dres.arg(), transpose_b=True, beta=1.0, b_scales=ds.arg())
    err = dout.download().astype(np.float64) - (exact - rounded.astype(np.float64))
    rel = np.sqrt(np.mean(err ** 2) / np.mean(exact ** 2)) * 2 ** 24
    assert rel <= np.sqrt(0.49 + 0.42 ** 2 * K / 16 / chains), rel
    for b in (dx, dw, ds, dres, dout):
        b.free()


@pytest.mark.parametrize("weights", ["f16", "q8", "q4"])
@pytest.mark.parametrize("K,H,Hkv,D,m,bs,layer", [
    (64, 3, 1, 64, 77, 16, 2),      # 64 x 64 (block-quantised 64 x 32): ragged rows and columns
    (128, 16, 2, 64, 1030, 48, 2),  # 128 x 64; pages that are not a power of two
    (64, 14, 2, 64, 2047, 16, 3),   # 128 x 128; a layer without a rotation
    (64, 40, 8, 64, 1000, 48, 2),   # 256 x 128: two turns of the write stage
    (192, 32, 4, 64, 520, 16, 2),   # 64 x 96: a third of a thread's pieces in each of three columns where steps are the waves' own
    (1024, 16, 2, 128, 524, 48, 2),
    (64, 24, 8, 128, 2040, 48, 2),  # F16: 256 x 160, five columns per thread, rows of two matrices
    (64, 24, 8, 128, 2048, 16, 3),
])
def test_write_stage_into_pages(K, H, Hkv, D, m, bs, layer, weights):
    """KvPrepFused as a tile's write stage against the two ops, bit for bit: pages, both pairings, with and without biases, layers
    that are not rotated (every fourth)."""
    announce("tiles, write stage into pages", K, H, Hkv, D, m, bs, layer, weights)
    f = ctx()
    rng = np.random.default_rng(K + H + m)
    N, NK, pos = H * D, Hkv * D, 37
    x, g, ws, bias = _data(rng, K, N, NK, m)
    if weights == "f16":
        dev, scales = [f.array(orc.to_canonical(w)) for w in ws], None
        arg = [w.arg() for w in dev]
    else:
        quant = [orc.quantize_q8_0(w) if weights == "q8" else orc.quantize_q4_0(w) for w in ws]
        flat = [orc.to_canonical(q) for q, _ in quant]
        dev = [f.array(q if weights == "q8" else orc.pack_q4_0(q)) for q in flat]
        arg = [w.arg() if weights == "q8" else w.arg((n, K), dtype=fa.DTYPE_Q4_0) for w, n in zip(dev, (N, NK, NK))]
        dev_s = [f.array(s) for _, s in quant]
        scales, dev = tuple(s.arg() for s in dev_s), dev + dev_s
    cos, sin = fa.rope_tables(1e6, D, pos + m)
    dx, dg, db, dcos, dsin = f.array(x), f.array(g), [f.array(b) for b in bias], f.array(cos), f.array(sin)
    outs, dqr = [f.zeros((m, n)) for n in (N, NK, NK)], [f.zeros((H, m, D)) for _ in range(2)]
    pgs = [Paged(f, np.random.default_rng(5), [0, pos, 0], Hkv, D, bs, extra_tokens=m + 1).upload() for _ in range(2)]
    try:
        f.set_gemm_min_m(12)
        for mode, biases in ((fa.ROPE_NEOX, tuple(b.arg() for b in db)), (fa.ROPE_NORMAL, None), (fa.ROPE_NORMAL, tuple(b.arg() for b in db))):
            kw = dict(gamma=dg.arg(), biases=biases, scales=scales)
            p = fa.KvPrepFusedParams.make(H, Hkv, D, m, pos, 0, mode, layer, 4)
            f.fused_qkv(dx.arg(), *arg, *[o.arg() for o in outs], K, N, NK, m, **kw)
            f.kv_prep_fused_paged(*[o.arg() for o in outs], dqr[0].arg(), pgs[0].desc, 1, dcos.arg(), dsin.arg(), p)
            f.fused_qkv_kv_prep(dx.arg(), *arg, K, dqr[1].arg(), dcos.arg(), dsin.arg(), p, paged=pgs[1].desc, seq_index=1, **kw)
            assert np.array_equal(bits(dqr[0].download()), bits(dqr[1].download())), mode
            for one, two in ((pgs[0].dk, pgs[1].dk), (pgs[0].dv, pgs[1].dv)):  # the whole pools: nothing is written beside the rows
                assert np.array_equal(bits(one.download()), bits(two.download())), mode
    finally:
        f.set_gemm_min_m()
        for pg in pgs:
            pg.free()
        for b in dev + db + outs + dqr + [dx, dg, dcos, dsin]:
            b.free()


@pytest.mark.parametrize("mode", [fa.ROPE_NORMAL, fa.ROPE_NEOX])
@pytest.mark.parametrize("H,Hkv,D,m", [(3, 1, 64, 77), (24, 8, 128, 2040)])  # a tile whose pieces are all asked for ahead, and 256 x 160
def test_rotation_of_the_smallest_and_largest_values(H, Hkv, D, m, mode):
    """KvPrepFused as a tile's write stage against the two ops where the projections are zeros of both signs, denormals, the largest
    values and infinities, and so are the tables: the same bits, a NaN wherever there is one."""
    announce("tiles, rotation of extreme values", H, Hkv, D, m, mode)
    f = ctx()
    rng = np.random.default_rng(H + m)
    K, N, NK = 64, H * D, Hkv * D
    values = np.array([0.0, -0.0, 6e-8, -6e-8, 1e-5, -1e-5, 0.333, -1.7, 300.0, 65504.0, -65504.0], np.float16)
    x = np.zeros((m, K), np.float16)  # one feature per row: the projections are that value times a weight
    x[np.arange(m), rng.integers(0, K, m)] = rng.choice(np.array([1.0, -1.0, 2.0, 0.25], np.float16), m)
    ws = [rng.choice(values, (n, K)) for n in (N, NK, NK)]
    cos, sin = (rng.choice(np.array([0.0, -0.0, 1.0, -1.0, 6e-8, 0.7, -1e-5], np.float16), (m + 3, D // 2)) for _ in range(2))
    dev, dx, dcos, dsin = [f.array(orc.to_canonical(w)) for w in ws], f.array(x), f.array(cos), f.array(sin)
    outs, dqr = [f.zeros((m, n)) for n in (N, NK, NK)], [f.zeros((H, m, D)) for _ in range(2)]
    kc, vc = ([f.zeros((Hkv, m + 3, D)) for _ in range(2)] for _ in range(2))
    try:
        f.set_gemm_min_m(12)
        p = fa.KvPrepFusedParams.make(H, Hkv, D, m, 3, m + 3, mode)
        f.fused_qkv(dx.arg(), *[w.arg() for w in dev], *[o.arg() for o in outs], K, N, NK, m)
        f.kv_prep_fused(*[o.arg() for o in outs], dqr[0].arg(), kc[0].arg(), vc[0].arg(), dcos.arg(), dsin.arg(), p)
        f.fused_qkv_kv_prep(dx.arg(), *[w.arg() for w in dev], K, dqr[1].arg(), dcos.arg(), dsin.arg(), p, k_cache=kc[1].arg(), v_cache=vc[1].arg())
        for one, two in (dqr, kc, vc):
            one, two = one.download(), two.download()
            assert np.array_equal(np.isnan(one), np.isnan(two))
            assert np.array_equal(bits(one)[~np.isnan(one)], bits(two)[~np.isnan(two)])
    finally:
        f.set_gemm_min_m()
        for b in dev + outs + dqr + kc + vc + [dx, dcos, dsin]:
            b.free()
