"""GPU: the attention kernel that gives 32 query rows to a workgroup (chunks and prompts of moderate size, the automatic choice)
against the oracle, at the edges of what it divides: rows of a KV group's heads in blocks of 32, keys in tiles of 32 over 4 or 8
waves, keys split over workgroups, pages."""
import numpy as np
import pytest

import foundry_attn as fa
import orc
from gpu_util import announce, ctx, h16, max_abs
from test_gpu_paged import Paged

pytestmark = pytest.mark.gpu
TOL, TOL_BF16 = 2e-3, 2e-2
BF = fa.DTYPE_BF16


def _launches(f, call):
    """What the call put on the stream: (this kernel, merge launches, any other attention kernel)."""
    f.profile_reset()
    f.profile_enable(True)
    try:
        call()
        f.synchronize()
        n = {k: f.profile_query(k)[0] for k in ("flash_rows_kernel", "flash_prefill_merge_kernel", "flash_")}
    finally:
        f.profile_enable(False)
    return n["flash_rows_kernel"], n["flash_prefill_merge_kernel"], n["flash_"] - n["flash_rows_kernel"] - n["flash_prefill_merge_kernel"]


CASES = [
    # H, Hkv, D, rows, prefix, splits expected
    (14, 2, 64, 2, 0, False),        # fewest rows: 14 of a block's 32
    (14, 2, 64, 4, 27, False),       # 28 rows of a block; 31 keys, one short of a tile
    (14, 2, 64, 5, 27, False),       # 35 rows: three of a second block; 32 keys
    (16, 2, 128, 4, 29, False),      # 32 rows: a whole block; 33 keys
    (4, 4, 128, 33, 64, False),      # a head to a group: one row of a second block
    (6, 2, 128, 17, 239, False),     # 256 keys: one tile per wave of eight
    (6, 2, 128, 17, 240, False),     # one key more
    (14, 2, 64, 100, 157, False),
    (24, 8, 128, 100, 700, False),
    (14, 2, 64, 500, 0, False),      # a prompt: every block another number of keys
    (14, 2, 64, 650, 31, False),     # more blocks than compute units: four waves
    (24, 8, 128, 401, 9, False),     # the same at D 128
    (12, 4, 64, 3, 3000, True),      # few rows, many keys: split
    (24, 8, 128, 20, 2900, True),
    (8, 2, 64, 32, 5001, True),
    (5, 1, 128, 7, 8161, True),      # one KV head
]


@pytest.mark.parametrize("bf16", [False, True], ids=["f16", "bf16"])
@pytest.mark.parametrize("H,Hkv,D,M,prefix,split", CASES)
def test_rows_contiguous(H, Hkv, D, M, prefix, split, bf16):
    announce("prefill rows", H, Hkv, D, M, prefix, split, bf16)
    f = ctx()
    rng = np.random.default_rng(M * 7 + prefix)
    N = prefix + M
    cap = N + 7
    q, k, v = (rng.normal(size=s).astype(np.float32) for s in ((H, M, D), (Hkv, cap, D), (Hkv, cap, D)))
    k[:, N:], v[:, N:] = np.nan, np.nan  # nothing past the visible keys is used
    conv = orc.bf16_pack if bf16 else h16
    q, k, v = conv(q), conv(k), conv(v)
    dt = BF if bf16 else fa.DTYPE_F16
    dq, dk, dv, do = (f.array(x) for x in (q, k, v, np.full((M, H * D), 0x7fc0 if bf16 else 0x7e00, np.uint16)))
    args = [b.arg(dtype=dt) for b in (dq, dk, dv, do)]
    n = _launches(f, lambda: f.flash_attention(*args, True, prefix, H, D, N, M))
    assert n == (1, 1 if split else 0, 0), n
    want = lambda: orc.sdpa_prefill(q, k, v, H, Hkv, D, M, N, prefix, cap, causal=True, out_layout="token_major", n_threads=8)
    raw = do.download()
    if bf16:
        with orc.bf16_mode():
            w = orc.bf16_unpack(want())
        got = orc.bf16_unpack(raw)
    else:
        w, got = want(), raw.view(np.float16)
    assert np.all(np.isfinite(got))
    assert max_abs(got.reshape(M, H * D), w.reshape(M, H * D)) <= (TOL_BF16 if bf16 else TOL)
    for b in (dq, dk, dv, do):
        b.free()


@pytest.mark.parametrize("bs", [16, 48, 64])
@pytest.mark.parametrize("H,Hkv,D,M,prefix,split", CASES[::2] + CASES[-4:-1])
def test_rows_paged(H, Hkv, D, M, prefix, split, bs):
    """Pages of one row group, of a number that is not a power of two, and of two tiles; the last page partly filled."""
    announce("prefill rows, paged", H, Hkv, D, M, prefix, split, bs)
    f = ctx()
    rng = np.random.default_rng(M * 11 + prefix + bs)
    N = prefix + M
    lens = [3, N]
    ks = [h16(rng.normal(size=(Hkv, n, D))) for n in lens]
    vs = [h16(rng.normal(size=(Hkv, n, D))) for n in lens]
    pg = Paged(f, rng, lens, Hkv, D, bs, extra_tokens=0)
    pg.fill_from(ks, vs)
    last = pg.bt[1, (N - 1) // bs]
    if N % bs:  # rows past the sequence's end, in its own last page
        pg.k_pool[last, :, N % bs:], pg.v_pool[last, :, N % bs:] = np.nan, np.nan
    pg.upload()
    q = h16(rng.normal(size=(H, M, D)))
    dq, do = f.array(q), f.zeros((M, H * D))
    n = _launches(f, lambda: f.flash_prefill_paged(dq.arg(), pg.desc, 1, do.arg(), True, prefix, H, N, M))
    assert n == (1, 1 if split else 0, 0), n
    got = do.download()
    want = orc.sdpa_prefill(q, ks[1], vs[1], H, Hkv, D, M, N, prefix, N, causal=True, n_threads=8)
    assert np.all(np.isfinite(got))
    assert max_abs(got.reshape(M, H * D), want.reshape(M, H * D)) <= TOL
    pg.free()
    for b in (dq, do):
        b.free()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("M,N,offset,causal", [(45, 300, 0, False), (45, 300, 3, True), (45, 60, 100, True), (9, 4000, 17, False)])
def test_rows_masks_and_layouts(M, N, offset, causal, D):
    """Without the causal mask; query positions in the middle of the keys and past their end; token-major queries and head-major
    output give the bits of the head-major queries and token-major output."""
    announce("prefill rows, masks and layouts", M, N, offset, causal, D)
    f = ctx()
    rng = np.random.default_rng(N + offset)
    H, Hkv, cap = 6, 2, N + 3
    q, k, v = h16(rng.normal(size=(H, M, D))), h16(rng.normal(size=(Hkv, cap, D))), h16(rng.normal(size=(Hkv, cap, D)))
    dk, dv = f.array(k), f.array(v)
    outs = []
    for token_major in (False, True):
        dq = f.array(np.ascontiguousarray(q.transpose(1, 0, 2)) if token_major else q)
        do = f.zeros((H, M, D) if token_major else (M, H * D))
        qa = dq.arg((M, H, D) if token_major else (H, M, D))
        n = _launches(f, lambda: f.flash_attention(qa, dk.arg(), dv.arg(), do.arg(), causal, offset, H, D, N, M))
        assert n[0] == 1 and n[2] == 0, n
        got = do.download()
        outs.append(got if token_major else got.reshape(M, H, D).transpose(1, 0, 2))
        dq.free(), do.free()
    assert np.array_equal(np.ascontiguousarray(outs[0]).view(np.uint16), outs[1].view(np.uint16))
    want = orc.sdpa_prefill(q, k, v, H, Hkv, D, M, N, offset, cap, causal=causal, out_layout="head_major", n_threads=8)
    assert max_abs(outs[1], want) <= TOL
    dk.free(), dv.free()


@pytest.mark.parametrize("D,M,prefix", [(64, 40, 2300), (128, 33, 1111), (64, 2, 40)])
def test_rows_paged_large_pool(D, M, prefix):
    """Pools of 4 GiB, whose rows have no 32-bit byte offsets, with pages all over them: the bits of the small pools' launch."""
    announce("prefill rows, large pool", D, M, prefix)
    f = ctx()
    rng = np.random.default_rng(D + M)
    H, Hkv, bs, N = 6, 2, 16, prefix + M
    nb = (N + bs - 1) // bs
    k, v, q0 = (f.array(h16(rng.normal(size=(N, h * D)))) for h in (Hkv, Hkv, H))
    q, q_rot = f.array(h16(rng.normal(size=(H, M, D)))), f.zeros((H, N, D))
    cos, sin = (f.array(t) for t in fa.rope_tables(1e4, D, N))
    lens, got = f.array(np.array([N], np.uint32)), []
    for n_pages in (nb + 3, 2 ** 32 // (Hkv * bs * D * 2)):
        table = rng.permutation(n_pages)[:nb].astype(np.int32)
        if n_pages - 1 not in table:
            table[-1] = n_pages - 1
        kp, vp, bt = f.empty((n_pages, Hkv, bs, D)), f.empty((n_pages, Hkv, bs, D)), f.array(table)
        cache = fa.paged_kv(kp, vp, bt, lens, n_pages, Hkv, bs, D, 1, nb)
        p = fa.KvPrepFusedParams.make(H, Hkv, D, N, 0, nb * bs, fa.ROPE_NEOX)
        f.kv_prep_fused_paged(q0.arg(), k.arg(), v.arg(), q_rot.arg(), cache, 0, cos.arg(), sin.arg(), p)
        do = f.zeros((M, H * D))
        n = _launches(f, lambda: f.flash_prefill_paged(q.arg(), cache, 0, do.arg(), True, prefix, H, N, M))
        assert n[0] == 1 and n[2] == 0, n
        got.append(do.download().view(np.uint16))
        for b in (kp, vp, bt, do):
            b.free()
    assert np.any(got[0]) and np.array_equal(got[0], got[1])
    for b in (k, v, q0, q, q_rot, cos, sin, lens):
        b.free()


@pytest.mark.parametrize("H,Hkv,D,M,prefix,bs", [(28, 2, 64, 300, 4500, 16), (32, 2, 64, 260, 4100, 48)])
def test_rows_paged_more_than_32_tiles_per_wave(H, Hkv, D, M, prefix, bs):
    """A wave fetches where its tiles lie a second time (4 waves)."""
    test_rows_paged(H, Hkv, D, M, prefix, False, bs)


TURNED = [
    # More than 4 MB of keys: blocks that share an XCD attend windows of rounds, each from a round of its own on
    # H, Hkv, D, rows, prefix, splits expected
    (24, 8, 128, 300, 950, False),   # windows of 4 or 8 rounds, the last one shorter; every block another number of keys
    (24, 8, 128, 300, 1020, False),
    (8, 8, 128, 66, 3001, True),     # 3 blocks, keys split: a window of 2 rounds, splits of unequal lengths
    (6, 2, 128, 200, 4100, True),    # two blocks of a KV head to an XCD, and three
    (16, 8, 128, 700, 400, False),   # several workgroups to a unit
    (16, 8, 64, 200, 2350, False),   # D 64
    (20, 5, 128, 120, 2000, False),  # KV heads that are not a divisor of 8: every eighth block of one is on the same XCD
]


@pytest.mark.parametrize("bf16", [False, True], ids=["f16", "bf16"])
@pytest.mark.parametrize("H,Hkv,D,M,prefix,split", TURNED)
def test_rows_turned_contiguous(H, Hkv, D, M, prefix, split, bf16):
    test_rows_contiguous(H, Hkv, D, M, prefix, split, bf16)


@pytest.mark.parametrize("bs", [16, 48])
@pytest.mark.parametrize("H,Hkv,D,M,prefix,split", TURNED + [(32, 2, 64, 620, 3700, False)])
def test_rows_turned_paged(H, Hkv, D, M, prefix, split, bs):
    """The last: several windows, and more than 32 tiles to a wave, whose pages are looked up a second time at a window's start."""
    test_rows_paged(H, Hkv, D, M, prefix, split, bs)


IN_TURNED_ORDERS = [
    # H, Hkv, D, rows, prefix, splits expected
    (24, 8, 128, 300, 950, False),   # one workgroup to a unit, four waves: windows of 8 rounds and a last one of fewer
    (24, 8, 128, 300, 1020, False),  # eight waves, windows of 4
    (20, 5, 128, 120, 2000, False),  # KV heads that are not a divisor of 8
    (8, 8, 128, 66, 3001, True),     # split: windows of 2
    (16, 8, 128, 700, 1500, False),  # several workgroups to a unit
    (32, 8, 64, 300, 5000, False),   # D 64, windows of 32 rounds, more than 32 tiles to a wave: pages are looked up a second time
]


def _turned():
    """Launches in turned orders since the profile was last reset."""
    return ctx().profile_query("flash_rows_kernel_turned")[0]


@pytest.mark.parametrize("bf16", [False, True], ids=["f16", "bf16"])
@pytest.mark.parametrize("H,Hkv,D,M,prefix,split", IN_TURNED_ORDERS)
def test_turned_orders_contiguous(H, Hkv, D, M, prefix, split, bf16):
    test_rows_contiguous(H, Hkv, D, M, prefix, split, bf16)
    assert _turned() == 1


@pytest.mark.parametrize("H,Hkv,D,M,prefix,split", [
    (6, 2, 128, 200, 4100, True),    # 4.4 MB of keys, split
    (14, 2, 64, 54, 15370, True),    # 7.9
    (16, 8, 128, 700, 400, False),   # 4.5, several workgroups to a unit
])
def test_one_order_of_fewer_keys(H, Hkv, D, M, prefix, split):
    """Between 4 MB and where turned orders are ahead of one for launches that are split or have several workgroups to a unit."""
    test_rows_contiguous(H, Hkv, D, M, prefix, split, False)
    assert _turned() == 0


@pytest.mark.parametrize("bs", [16, 48])
@pytest.mark.parametrize("H,Hkv,D,M,prefix,split", IN_TURNED_ORDERS)
def test_turned_orders_paged(H, Hkv, D, M, prefix, split, bs):
    test_rows_paged(H, Hkv, D, M, prefix, split, bs)
    assert _turned() == 1


def test_turned_orders_large_pool():
    test_rows_paged_large_pool(128, 100, 9000)
    assert _turned() == 1


@pytest.mark.parametrize("M,N,offset,causal", [(200, 9300, 0, False), (200, 9300, 9400, True)])
def test_turned_orders_masks(M, N, offset, causal):
    """Without the causal mask; query positions past the keys' end."""
    test_rows_masks_and_layouts(M, N, offset, causal, 128)
    assert _turned() == 1


@pytest.mark.parametrize("H,Hkv,D,M,prefix", [(24, 8, 128, 278, 7179), (16, 2, 128, 34, 47550), (32, 8, 128, 51, 19165), (4, 4, 128, 18, 44996)])
def test_long_keys_from_memory_stay_with_the_other_kernels(H, Hkv, D, M, prefix):
    """Shapes that take 1.15 to 1.6 times as long on this kernel where their keys come from memory: the choice is another one, with its
    result (two orders of the same sums: an f16 ulp)."""
    announce("prefill rows, long keys", H, Hkv, D, M, prefix)
    f = ctx()
    rng = np.random.default_rng(M + prefix)
    N = prefix + M
    k, v = (h16(np.resize(rng.normal(size=1000003), (Hkv, N, D))) for _ in range(2))
    dq, dk, dv, do = f.array(h16(rng.normal(size=(H, M, D)))), f.array(k), f.array(v), f.zeros((M, H * D))

    def call():
        f.flash_attention(dq.arg(), dk.arg(), dv.arg(), do.arg(), True, prefix, H, D, N, M)

    n = _launches(f, call)
    assert n[0] == 0 and n[2] == 1, n
    got = do.download()
    f.set_prefill_variant(2)
    try:
        call()
    finally:
        f.set_prefill_variant(0)
    assert np.any(got) and max_abs(got, do.download()) <= TOL
    for b in (dq, dk, dv, do):
        b.free()
