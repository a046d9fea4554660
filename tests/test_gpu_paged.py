"""GPU parity: paged KV cache (block table, per-sequence lengths). The reference has no paged cache; the
contract is gather(paged) == the contiguous cache the reference would hold, bit for bit, and attention over
the paged cache == attention over that contiguous cache."""
import numpy as np
import pytest

import foundry_attn as fa
import orc
from gpu_util import announce, bits, ctx, h16, max_abs

pytestmark = pytest.mark.gpu
TOL = 2e-3


class Paged:
    """Host mirror of a paged pool with a seeded random permutation of physical blocks."""

    def __init__(self, f, rng, lens, Hkv, D, bs, extra_tokens=1, slack_blocks=3):
        self.f, self.Hkv, self.D, self.bs = f, Hkv, D, bs
        self.lens = np.asarray(lens, np.uint32)
        self.n_seqs = len(lens)
        need = [(int(n) + extra_tokens + bs - 1) // bs for n in lens]
        self.mb = max(need)
        self.n_blocks = sum(need) + slack_blocks
        perm = rng.permutation(self.n_blocks).astype(np.int32)
        self.bt = np.full((self.n_seqs, self.mb), -1, np.int32)
        o = 0
        for s, n in enumerate(need):
            self.bt[s, :n] = perm[o:o + n]
            o += n
        self.bt_dev_host = np.where(self.bt < 0, 0, self.bt).astype(np.int32)
        self.k_pool = np.zeros((self.n_blocks, Hkv, bs, D), np.float16)
        self.v_pool = np.zeros((self.n_blocks, Hkv, bs, D), np.float16)

    def fill_from(self, ks, vs):
        for s in range(self.n_seqs):
            orc.paged_scatter(self.k_pool, self.bt[s], self.Hkv, self.bs, self.D, 0, int(self.lens[s]), ks[s])
            orc.paged_scatter(self.v_pool, self.bt[s], self.Hkv, self.bs, self.D, 0, int(self.lens[s]), vs[s])

    def upload(self):
        f = self.f
        self.dk, self.dv = f.array(self.k_pool), f.array(self.v_pool)
        self.dbt, self.dlens = f.array(self.bt_dev_host), f.array(self.lens)
        self.desc = fa.paged_kv(self.dk, self.dv, self.dbt, self.dlens, self.n_blocks, self.Hkv, self.bs, self.D,
                                self.n_seqs, self.mb)
        return self

    def free(self):
        for b in (self.dk, self.dv, self.dbt, self.dlens):
            b.free()


@pytest.mark.parametrize("H,Hkv,D,bs,lens", [
    (16, 2, 128, 16, [512, 777, 16, 1, 4095, 1000, 33, 2049]),   # Qwen2.5-3B shape (benchmark configuration 3), ragged
    (14, 2, 64, 16, [100, 5, 64]),
    (24, 8, 128, 32, [300, 31]),
    (8, 8, 64, 64, [129]),
    (24, 8, 128, 16, [40000]),  # one long sequence: whole partitions, one per compute unit, merged inside the launch
])
def test_paged_batched_decode_step(H, Hkv, D, bs, lens):
    """One batched decode step: append one token per sequence at seq_lens[b], then ragged flash decode."""
    announce("paged decode step", H, Hkv, D, bs, lens)
    f = ctx()
    rng = np.random.default_rng(len(lens) * 100 + D)
    B = len(lens)
    ks = [h16(rng.normal(size=(Hkv, n + 1, D))) for n in lens]
    vs = [h16(rng.normal(size=(Hkv, n + 1, D))) for n in lens]
    pg = Paged(f, rng, lens, Hkv, D, bs)
    pg.fill_from(ks, vs)
    pg.upload()
    q = h16(rng.normal(size=(B, H * D)))
    kn = h16(rng.normal(size=(B, Hkv * D)))
    vn = h16(rng.normal(size=(B, Hkv * D)))
    maxpos = int(max(lens)) + 1
    cos, sin = fa.rope_tables(1e6, D, maxpos)
    dq, dkn, dvn, dqr, dout = f.array(q), f.array(kn), f.array(vn), f.zeros((B, H, D)), f.zeros((B, H * D))
    dcos, dsin = f.array(cos), f.array(sin)
    p = fa.KvPrepFusedParams.make(H, Hkv, D, B, 0, 0, fa.ROPE_NEOX)
    f.kv_prep_decode_paged(dq.arg(), dkn.arg(), dvn.arg(), dqr.arg(), pg.desc, dcos.arg(), dsin.arg(), p)
    f.flash_decode_paged(dqr.arg(), pg.desc, dout.arg(), H, 1, maxpos)
    f.synchronize()
    got_qr, got_out = dqr.download(), dout.download().reshape(B, H, D)
    got_kp, got_vp = pg.dk.download(), pg.dv.download()
    gk, gv = f.zeros((Hkv, maxpos, D)), f.zeros((Hkv, maxpos, D))
    for b, n in enumerate(lens):
        # oracle: the reference's contiguous cache after the same append
        kc = np.zeros((Hkv, n + 1, D), np.float16)
        vc = np.zeros((Hkv, n + 1, D), np.float16)
        kc[:, :n], vc[:, :n] = ks[b][:, :n], vs[b][:, :n]
        want_qr = orc.kv_prep_fused(q[b:b + 1], kn[b:b + 1], vn[b:b + 1], kc, vc, cos, sin,
                                    orc.make_params(H, Hkv, D, 1, n, n + 1, rope_mode=0))
        assert np.array_equal(bits(got_qr[b]), bits(want_qr[:, 0])), b
        # host-side gather of the downloaded pools and the device gather kernel agree with it bit for bit
        assert np.array_equal(bits(orc.paged_gather(got_kp, pg.bt[b], Hkv, bs, D, n + 1)), bits(kc)), b
        assert np.array_equal(bits(orc.paged_gather(got_vp, pg.bt[b], Hkv, bs, D, n + 1)), bits(vc)), b
        f.paged_gather(pg.desc, b, n + 1, gk, gv, maxpos)
        f.synchronize()
        assert np.array_equal(bits(gk.download()[:, :n + 1]), bits(kc)), b
        assert np.array_equal(bits(gv.download()[:, :n + 1]), bits(vc)), b
        want = orc.sdpa_decode(want_qr[:, 0].copy(), kc, vc, H, Hkv, D, n + 1, n + 1).reshape(H, D)
        assert max_abs(got_out[b], want) <= TOL, b
    # blocks outside every block table were not touched
    used = set(pg.bt[pg.bt >= 0].tolist())
    for blk in range(pg.n_blocks):
        if blk not in used:
            assert not got_kp[blk].any() and not got_vp[blk].any()
    pg.free()
    for b in (dq, dkn, dvn, dqr, dout, dcos, dsin, gk, gv):
        b.free()


@pytest.mark.usefixtures("prefill_variant")
def test_paged_prefill_append_then_decode_equals_contiguous():
    """Multi-token append into an empty paged cache (one sequence of a batch), compared with the contiguous op."""
    announce("paged prefill append")
    f = ctx()
    rng = np.random.default_rng(77)
    H, Hkv, D, bs, T = 24, 8, 128, 16, 150
    pg = Paged(f, rng, [0, 0, 0], Hkv, D, bs, extra_tokens=T + 1).upload()
    q, k, v = (h16(rng.normal(size=(T, n * D))) for n in (H, Hkv, Hkv))
    cos, sin = fa.rope_tables(5e5, D, 256)
    dq, dk, dv, dqr = f.array(q), f.array(k), f.array(v), f.zeros((H, T, D))
    dcos, dsin = f.array(cos), f.array(sin)
    p = fa.KvPrepFusedParams.make(H, Hkv, D, T, 0, 0, fa.ROPE_NORMAL)
    f.kv_prep_fused_paged(dq.arg(), dk.arg(), dv.arg(), dqr.arg(), pg.desc, 1, dcos.arg(), dsin.arg(), p)
    f.synchronize()
    kc, vc = np.zeros((Hkv, T, D), np.float16), np.zeros((Hkv, T, D), np.float16)
    want_qr = orc.kv_prep_fused(q, k, v, kc, vc, cos, sin, orc.make_params(H, Hkv, D, T, 0, T, rope_mode=1))
    assert np.array_equal(bits(dqr.download()), bits(want_qr))
    assert np.array_equal(bits(orc.paged_gather(pg.dk.download(), pg.bt[1], Hkv, bs, D, T)), bits(kc))
    assert np.array_equal(bits(orc.paged_gather(pg.dv.download(), pg.bt[1], Hkv, bs, D, T)), bits(vc))
    # sequences 0 and 2 own other blocks: still empty
    for s in (0, 2):
        assert not orc.paged_gather(pg.dk.download(), pg.bt[s], Hkv, bs, D, T).any()
    with pytest.raises(fa.FoundryError) as e:  # beyond the block table
        f.kv_prep_fused_paged(dq.arg(), dk.arg(), dv.arg(), dqr.arg(), pg.desc, 1, dcos.arg(), dsin.arg(),
                              fa.KvPrepFusedParams.make(H, Hkv, D, T, pg.mb * bs - 3, 0, fa.ROPE_NORMAL))
    assert e.value.variant == "InvalidOperation"
    with pytest.raises(fa.FoundryError) as e:
        f.kv_prep_fused_paged(dq.arg(), dk.arg(), dv.arg(), dqr.arg(), pg.desc, 3, dcos.arg(), dsin.arg(), p)
    assert e.value.variant == "InvalidShape"
    f.synchronize()
    pg.free()


def test_paged_decode_multi_step_advances_lengths():
    """Three decode steps with device-side length advance between them (fa_u32_add)."""
    announce("paged multi-step")
    f = ctx()
    rng = np.random.default_rng(5)
    H, Hkv, D, bs, steps = 16, 2, 128, 16, 3
    lens = [30, 47, 16]
    B = len(lens)
    ks = [h16(rng.normal(size=(Hkv, n + steps, D))) for n in lens]
    vs = [h16(rng.normal(size=(Hkv, n + steps, D))) for n in lens]
    pg = Paged(f, rng, lens, Hkv, D, bs, extra_tokens=steps)
    pg.fill_from(ks, vs)
    pg.upload()
    cos, sin = fa.rope_tables(1e6, D, 128)
    dcos, dsin = f.array(cos), f.array(sin)
    kc = [np.zeros((Hkv, n + steps, D), np.float16) for n in lens]
    vc = [np.zeros((Hkv, n + steps, D), np.float16) for n in lens]
    for b, n in enumerate(lens):
        kc[b][:, :n], vc[b][:, :n] = ks[b][:, :n], vs[b][:, :n]
    dqr, dout = f.zeros((B, H, D)), f.zeros((B, H * D))
    p = fa.KvPrepFusedParams.make(H, Hkv, D, B, 0, 0, fa.ROPE_NEOX)
    for t in range(steps):
        q, kn, vn = (h16(rng.normal(size=(B, n * D))) for n in (H, Hkv, Hkv))
        dq, dkn, dvn = f.array(q), f.array(kn), f.array(vn)
        f.kv_prep_decode_paged(dq.arg(), dkn.arg(), dvn.arg(), dqr.arg(), pg.desc, dcos.arg(), dsin.arg(), p)
        f.flash_decode_paged(dqr.arg(), pg.desc, dout.arg(), H, 1, 64)
        f.u32_add(pg.dlens, B, 1)
        f.synchronize()
        got = dout.download().reshape(B, H, D)
        for b, n in enumerate(lens):
            qr = orc.kv_prep_fused(q[b:b + 1], kn[b:b + 1], vn[b:b + 1], kc[b], vc[b], cos, sin,
                                   orc.make_params(H, Hkv, D, 1, n + t, n + steps, rope_mode=0))
            want = orc.sdpa_decode(qr[:, 0].copy(), kc[b], vc[b], H, Hkv, D, n + steps, n + t + 1).reshape(H, D)
            assert max_abs(got[b], want) <= TOL, (t, b)
    assert np.array_equal(pg.dlens.download(), np.asarray(lens, np.uint32) + steps)
    pg.free()


def test_paged_fused_step_equals_separate_ops():
    """fa_decode_step_fused_paged == fa_kv_prep_decode_paged + fa_flash_decode_paged: q_rot and pools bit-identical,
    outputs equal up to f32 summation order."""
    announce("paged fused step")
    f = ctx()
    rng = np.random.default_rng(17)
    H, Hkv, D, bs = 16, 2, 128, 16
    lens = [512, 15, 16, 1, 1000, 63, 64, 0]
    B = len(lens)
    ks = [h16(rng.normal(size=(Hkv, n + 1, D))) for n in lens]
    vs = [h16(rng.normal(size=(Hkv, n + 1, D))) for n in lens]
    q, kn, vn = (h16(rng.normal(size=(B, n * D))) for n in (H, Hkv, Hkv))
    cos, sin = fa.rope_tables(1e6, D, 1024)
    dcos, dsin = f.array(cos), f.array(sin)
    dq, dkn, dvn = f.array(q), f.array(kn), f.array(vn)
    p = fa.KvPrepFusedParams.make(H, Hkv, D, B, 0, 0, fa.ROPE_NEOX)
    outs = []
    for fused in (False, True):
        pg = Paged(f, np.random.default_rng(3), lens, Hkv, D, bs)
        pg.fill_from(ks, vs)
        pg.upload()
        dqr, dout = f.zeros((B, H, D)), f.zeros((B, H * D))
        if fused:
            f.decode_step_fused_paged(dq.arg(), dkn.arg(), dvn.arg(), dqr.arg(), pg.desc, dcos.arg(), dsin.arg(),
                                      dout.arg(), p, 1024)
        else:
            f.kv_prep_decode_paged(dq.arg(), dkn.arg(), dvn.arg(), dqr.arg(), pg.desc, dcos.arg(), dsin.arg(), p)
            f.flash_decode_paged(dqr.arg(), pg.desc, dout.arg(), H, 1, 1024)
        f.synchronize()
        outs.append((dqr.download(), dout.download(), pg.dk.download(), pg.dv.download()))
        pg.free()
    for i, (a, b) in enumerate(zip(outs[0], outs[1])):
        if i == 1:
            assert max_abs(a, b) <= 2e-3
        else:
            assert np.array_equal(bits(a), bits(b))
    # and against the oracle for two of the sequences
    for b in (0, 7):
        n = lens[b]
        kc, vc = np.zeros((Hkv, n + 1, D), np.float16), np.zeros((Hkv, n + 1, D), np.float16)
        kc[:, :n], vc[:, :n] = ks[b][:, :n], vs[b][:, :n]
        qr = orc.kv_prep_fused(q[b:b + 1], kn[b:b + 1], vn[b:b + 1], kc, vc, cos, sin,
                               orc.make_params(H, Hkv, D, 1, n, n + 1, rope_mode=0))
        want = orc.sdpa_decode(qr[:, 0].copy(), kc, vc, H, Hkv, D, n + 1, n + 1).reshape(H, D)
        assert max_abs(outs[1][1].reshape(B, H, D)[b], want) <= TOL


def test_paged_decode_full_batch_of_32_ragged_sequences():
    """The Qwen2.5-3B-shaped batched paged decode at full size: 32 sequences with lengths drawn from 512..16384,
    16-token blocks behind a random block permutation. Every sequence against the oracle over its gathered cache."""
    announce("paged decode, 32 ragged sequences")
    f = ctx()
    rng = np.random.default_rng(2024)
    H, Hkv, D, bs, B = 16, 2, 128, 16, 32
    lens = [int(x) for x in rng.integers(512, 16385, size=B)]
    ks = [h16(rng.normal(size=(Hkv, n, D))) for n in lens]
    vs = [h16(rng.normal(size=(Hkv, n, D))) for n in lens]
    pg = Paged(f, rng, lens, Hkv, D, bs, extra_tokens=0)
    pg.fill_from(ks, vs)
    pg.upload()
    q = h16(rng.normal(size=(B, H, D)))
    dq, dout = f.array(q), f.zeros((B, H * D))
    f.flash_decode_paged(dq.arg(), pg.desc, dout.arg(), H, 0, max(lens))
    f.synchronize()
    got = dout.download().reshape(B, H, D)
    assert np.all(np.isfinite(got))
    worst = 0.0
    for b, n in enumerate(lens):
        want = orc.sdpa_decode(q[b], ks[b], vs[b], H, Hkv, D, n, n, n_threads=8).reshape(H, D)
        worst = max(worst, max_abs(got[b], want))
    print("32 ragged sequences, %d keys in total: max abs err %.2e" % (sum(lens), worst), flush=True)
    assert worst <= TOL
    pg.free()
    for b in (dq, dout):
        b.free()


@pytest.mark.parametrize("H,Hkv,D,bs,lens,bound", [
    (16, 2, 128, 16, [0, 4999], 0),                                             # one sequence has all the slots, at most 64 each
    (16, 2, 128, 16, [1, 15, 16, 17, 31, 0, 2047, 2048, 2049, 6000] * 3, 0),    # block edges, sequences of the new token alone
    (24, 8, 128, 32, [4000, 127, 128, 129, 2500, 3999, 1000, 64], 4096),        # 32 slots, an XCD's worth per KV head
    (8, 8, 128, 16, [100 + 97 * i for i in range(32)], 0),                      # two slots per sequence, four waves
    (6, 3, 128, 48, [3000, 10, 700, 1500], 0),                                  # 85 slots per head group: not dealt by XCD
    (14, 2, 64, 16, [(i * 977) % 4100 for i in range(64)], 0),                  # 64 sequences, every lane of the wave
    (16, 1, 128, 16, [5000, 3, 2222], 8192),                                    # 16 heads per workgroup, 256 slots
    (16, 2, 128, 16, [200, 30, 90, 155, 64, 12], 16384),                        # a bound far above the lengths
    # about equal lengths, dealt evenly: 16 slots each on an XCD of their own half, 5 each with slots left over, a length of none
    (16, 2, 128, 16, [8200 + 7 * i for i in range(8)], 0),
    (16, 2, 128, 16, [2600 + 3 * i for i in range(23)] + [0], 4096),
    (24, 8, 128, 16, [2000] * 7 + [2047], 0),
    (6, 3, 128, 48, [3000] * 5, 9216),                                          # ... and not by XCD
])
def test_paged_batch_dealt_out_by_lengths(H, Hkv, D, bs, lens, bound):
    """The launch whose workgroups find their (sequence, partition) from the lengths: against the oracle, and against the
    partitions cut by the bound with the merge in a second launch. The two add the same f32 partial sums in another grouping
    and round once to f16: two f16 units of the largest output apart at most."""
    announce("paged batch dealt out by lengths", H, Hkv, D, bs, len(lens), max(lens), bound)
    f = ctx()
    rng = np.random.default_rng(H + 10 * D + len(lens))
    B = len(lens)
    ks = [h16(rng.normal(size=(Hkv, n + 1, D))) for n in lens]
    vs = [h16(rng.normal(size=(Hkv, n + 1, D))) for n in lens]
    pg = Paged(f, rng, lens, Hkv, D, bs)
    if bound:  # (the launch's bound is cut to the block table's width)
        pg.mb = (bound + bs - 1) // bs
        wide = np.zeros((B, pg.mb), np.int32)
        wide[:, :pg.bt_dev_host.shape[1]] = pg.bt_dev_host
        pg.bt_dev_host = wide
    pg.fill_from(ks, vs)
    pg.upload()
    bound = bound or max(lens) + 1
    q, kn, vn = (h16(rng.normal(size=(B, n * D))) for n in (H, Hkv, Hkv))
    cos, sin = fa.rope_tables(1e6, D, max(lens) + 1)
    dq, dkn, dvn, dcos, dsin = f.array(q), f.array(kn), f.array(vn), f.array(cos), f.array(sin)
    p = fa.KvPrepFusedParams.make(H, Hkv, D, B, 0, 0, fa.ROPE_NEOX)
    outs, rots, pools = [], [], []
    for merge in (2, 2, 1):  # (twice: the exchange buffer is ready for the next launch)
        dout, dqr = f.zeros((B, H * D)), f.zeros((B, H, D))
        try:
            f.set_decode_variant(0, merge)
            f.decode_step_fused_paged(dq.arg(), dkn.arg(), dvn.arg(), dqr.arg(), pg.desc, dcos.arg(), dsin.arg(), dout.arg(), p, bound)
            f.synchronize()
        finally:
            f.set_decode_variant()
        outs.append(dout.download().reshape(B, H, D)), rots.append(dqr.download())
        pools.append((pg.dk.download(), pg.dv.download()))
        dout.free(), dqr.free()
    assert np.array_equal(bits(outs[0]), bits(outs[1]))
    for i in (0, 1):
        assert np.array_equal(bits(rots[i]), bits(rots[2]))
        assert all(np.array_equal(bits(x), bits(y)) for x, y in zip(pools[i], pools[2]))
    for b, n in enumerate(lens):
        unit = 2.0 ** (np.floor(np.log2(np.abs(outs[2][b].astype(np.float32)).max())) - 10)
        assert max_abs(outs[0][b], outs[2][b]) <= 2 * unit, b
        kc, vc = np.zeros((Hkv, n + 1, D), np.float16), np.zeros((Hkv, n + 1, D), np.float16)
        kc[:, :n], vc[:, :n] = ks[b][:, :n], vs[b][:, :n]
        qr = orc.kv_prep_fused(q[b:b + 1], kn[b:b + 1], vn[b:b + 1], kc, vc, cos, sin, orc.make_params(H, Hkv, D, 1, n, n + 1, rope_mode=0))
        want = orc.sdpa_decode(qr[:, 0].copy(), kc, vc, H, Hkv, D, n + 1, n + 1, n_threads=8).reshape(H, D)
        assert max_abs(outs[0][b], want) <= TOL, b
    pg.free()
    for x in (dq, dkn, dvn, dcos, dsin):
        x.free()


def widen(pg, bound):
    """A block table of `bound` tokens per sequence (a launch's bound is cut to the table's width)."""
    wide = np.zeros((pg.n_seqs, (bound + pg.bs - 1) // pg.bs), np.int32)
    wide[:, :pg.mb] = pg.bt_dev_host
    pg.bt_dev_host, pg.mb = wide, wide.shape[1]


@pytest.mark.parametrize("H,Hkv,D,B", [
    (16, 2, 128, 32),   # eight-wave workgroups
    (16, 2, 128, 60),   # four-wave workgroups
    (24, 8, 64, 12),
])
def test_paged_batch_that_does_not_fit_at_once_waits_for_nobody(H, Hkv, D, B):
    """A batch with more partitions by its bound than fit the GPU at once is merged without any workgroup waiting for another, also
    where its partitions are dealt out by the lengths: it is right on a GPU that it shares, here with a wait bound of zero (a launch
    whose workgroups wait would give up)."""
    announce("paged batch, zero wait bound", H, Hkv, D, B)
    rng = np.random.default_rng(B)
    lens = [int(x) for x in rng.integers(1, 700, size=B)]
    lens[1], bs, bound = 3000, 16, 16384
    ks = [h16(rng.normal(size=(Hkv, n, D))) for n in lens]
    vs = [h16(rng.normal(size=(Hkv, n, D))) for n in lens]
    q = h16(rng.normal(size=(B, H, D)))
    g = fa.Foundry(0)
    try:
        pg = Paged(g, rng, lens, Hkv, D, bs, extra_tokens=0)
        widen(pg, bound)
        pg.fill_from(ks, vs)
        pg.upload()
        dq, dout = g.array(q), g.zeros((B, H * D))
        g.set_decode_poll_spin_us(0)
        for _ in range(4):
            dout.upload(np.zeros((B, H * D), np.float16))
            g.flash_decode_paged(dq.arg(), pg.desc, dout.arg(), H, 0, bound)
            g.synchronize()
            got = dout.download().reshape(B, H, D)
            for b, n in enumerate(lens):
                want = orc.sdpa_decode(q[b], ks[b], vs[b], H, Hkv, D, n, n, n_threads=8).reshape(H, D)
                assert max_abs(got[b], want) <= TOL, b
    finally:
        g.close()


class Batch:
    """A fused decode step of a paged batch: inputs on the device, and per sequence the contiguous cache that it amounts to."""

    def __init__(self, f, rng, H, Hkv, D, bs, lens, mode, bf16=False, bound=0, extra=1):
        pack = orc.bf16_pack if bf16 else h16
        self.f, self.H, self.Hkv, self.D, self.lens, self.mode, self.bf16 = f, H, Hkv, D, list(lens), mode, bf16
        self.kc, self.vc = ([pack(rng.normal(size=(Hkv, n + extra, D))) for n in lens] for _ in range(2))
        self.pg = Paged(f, rng, lens, Hkv, D, bs, extra_tokens=extra)
        if bound:
            widen(self.pg, bound)
        for s in range(len(lens)):  # (rows past a sequence's length as well: they are overwritten as it grows)
            orc.paged_scatter(self.pg.k_pool, self.pg.bt[s], Hkv, bs, D, 0, lens[s] + extra, self.kc[s])
            orc.paged_scatter(self.pg.v_pool, self.pg.bt[s], Hkv, bs, D, 0, lens[s] + extra, self.vc[s])
        self.pg.upload()
        self.q, self.kn, self.vn = (pack(rng.normal(size=(len(lens), n * D))) for n in (H, Hkv, Hkv))
        self.cos, self.sin = fa.rope_tables(1e6, D, max(lens) + extra)
        self.dev = [f.array(x) for x in (self.q, self.kn, self.vn, self.cos, self.sin)]
        self.dqr, self.dout = f.zeros((len(lens), H, D)), f.zeros((len(lens), H * D))
        self.p = fa.KvPrepFusedParams.make(H, Hkv, D, len(lens), 0, 0, mode)
        self.bound = bound or max(lens) + extra

    def step(self):
        kw = dict(dtype=fa.DTYPE_BF16) if self.bf16 else {}
        dq, dkn, dvn, dcos, dsin = self.dev
        self.f.decode_step_fused_paged(dq.arg(**kw), dkn.arg(**kw), dvn.arg(**kw), self.dqr.arg(**kw), self.pg.desc, dcos.arg(), dsin.arg(),
                                       self.dout.arg(**kw), self.p, self.bound)

    def value(self, x):
        return orc.bf16_unpack(x) if self.bf16 else x

    def out(self):
        return self.value(self.dout.download()).reshape(len(self.lens), self.H, self.D)

    def want(self, b, n):
        """The oracle's step of sequence b at length n: appends to its contiguous cache, returns (q_rot, output)."""
        def go():
            cap = self.kc[b].shape[1]
            qr = orc.kv_prep_fused(self.q[b:b + 1], self.kn[b:b + 1], self.vn[b:b + 1], self.kc[b], self.vc[b], self.cos, self.sin,
                                   orc.make_params(self.H, self.Hkv, self.D, 1, n, cap, rope_mode=self.mode))
            return qr[:, 0].copy(), self.value(orc.sdpa_decode(qr[:, 0].copy(), self.kc[b], self.vc[b], self.H, self.Hkv, self.D, cap, n + 1,
                                                               n_threads=8)).reshape(self.H, self.D)
        if self.bf16:
            with orc.bf16_mode():
                return go()
        return go()

    def caches_match(self, b):
        n = self.kc[b].shape[1]
        return all(np.array_equal(bits(orc.paged_gather(d.download(), self.pg.bt[b], self.Hkv, self.pg.bs, self.D, n)), bits(c))
                   for d, c in ((self.pg.dk, self.kc[b]), (self.pg.dv, self.vc[b])))

    def free(self):
        self.pg.free()
        for x in self.dev + [self.dqr, self.dout]:
            x.free()


@pytest.mark.parametrize("bf16,mode", [(False, fa.ROPE_NORMAL), (True, fa.ROPE_NEOX), (True, fa.ROPE_NORMAL)])
@pytest.mark.parametrize("H,Hkv,D,lens", [
    (16, 2, 128, [1, 15, 16, 17, 31, 0, 2047, 2048, 2049, 5000] * 2),  # one after the other
    (24, 8, 128, [2000] * 7 + [2047]),                                # evenly
    (14, 2, 64, [(i * 977) % 2100 for i in range(40)]),
])
def test_paged_batch_dealt_out_by_lengths_types_and_pairings(H, Hkv, D, lens, bf16, mode):
    announce("paged batch dealt out by lengths", "bf16" if bf16 else "f16", mode, H, Hkv, D, len(lens))
    f = ctx()
    b = Batch(f, np.random.default_rng(H + D + mode), H, Hkv, D, 16, lens, mode, bf16)
    try:
        f.set_decode_variant(0, 2)
        b.step()
        f.synchronize()
    finally:
        f.set_decode_variant()
    got, rot = b.out(), b.dqr.download()
    for i, n in enumerate(lens):
        qr, want = b.want(i, n)
        assert np.array_equal(bits(rot[i]), bits(qr)) and b.caches_match(i), i
        assert max_abs(got[i], want) <= (1.6e-2 if bf16 else TOL), i  # (bf16: the bar of test_gpu_bf16.py)
    b.free()


@pytest.mark.parametrize("merge", [0, 2])
@pytest.mark.parametrize("H,Hkv,D,lens,bound,grow,steps", [
    (16, 2, 128, [200, 90, 0, 155, 64, 12], 4096, 301, 12),      # other partitions at every replay
    (24, 8, 128, [100 + 3 * i for i in range(8)], 2048, 157, 12),  # evenly, from a few keys each to the whole bound
    (14, 2, 64, [127] * 20 + [900], 0, 1, 3),                    # a block edge, the last token at the bound
])
def test_paged_batch_in_a_graph_as_its_lengths_grow(H, Hkv, D, lens, bound, grow, steps, merge):
    """One recorded step replayed while the lengths on the device grow: every replay against the oracle."""
    announce("paged batch in a graph, growing lengths", H, Hkv, D, len(lens), bound, grow, merge)
    f = ctx()
    extra = grow * (steps - 1) + 1
    b = Batch(f, np.random.default_rng(H + D), H, Hkv, D, 16, lens, fa.ROPE_NEOX, bound=bound, extra=extra)
    assert max(lens) + extra <= b.bound
    try:
        f.set_decode_variant(0, merge)
        b.step()  # eager: the workspace at its final size (and the rows that the first replay writes again)
        f.synchronize()
        f.start_capture()
        b.step()
        f.u32_add(b.pg.dlens, len(lens), grow)
        graph = f.end_capture()
    finally:
        f.set_decode_variant()
    for t in range(steps):
        b.dout.upload(np.zeros(b.dout.shape, np.float16))
        graph.launch()
        f.synchronize()
        got = b.out()
        for i, n in enumerate(lens):
            assert max_abs(got[i], b.want(i, n + t * grow)[1]) <= TOL, (t, i)
    assert all(b.caches_match(i) for i in range(len(lens)))
    graph.destroy()
    b.free()


def test_paged_batch_with_a_sequence_past_its_bound():
    """A sequence whose position lies past the launch's bound is not appended, the others are served, and the next wait reports it:
    the same whether the partitions are dealt out by the lengths or cut by the bound."""
    announce("paged batch, a sequence past the bound")
    g = fa.Foundry(0)
    try:
        H, Hkv, D, lens, bound = 16, 2, 128, [700, 30, 1024, 500, 1023, 999], 1024
        outs, pools = [], []
        for merge in (2, 1):
            b = Batch(g, np.random.default_rng(4), H, Hkv, D, 16, lens, fa.ROPE_NEOX, bound=1040)
            b.bound = bound
            before = b.pg.dk.download()
            g.set_decode_variant(0, merge)
            b.step()
            with pytest.raises(fa.FoundryError) as e:
                g.synchronize()
            assert e.value.variant == "InvalidOperation" and "neither appended nor attended" in str(e.value)
            g.synchronize()  # nothing is left over
            outs.append(b.out()), pools.append((b.pg.dk.download(), b.pg.dv.download()))
            for i, n in enumerate(lens):
                if n == bound:
                    rows = [orc.paged_gather(x, b.pg.bt[i], Hkv, 16, D, n + 1) for x in (before, pools[-1][0])]
                    assert np.array_equal(bits(rows[0]), bits(rows[1]))
                else:
                    want = b.want(i, n)[1]
                    assert b.caches_match(i) and max_abs(outs[-1][i], want) <= TOL, i
            b.free()
        assert all(np.array_equal(bits(x), bits(y)) for x, y in zip(*pools))
        assert max_abs(outs[0], outs[1]) <= TOL
    finally:
        g.close()


def test_polled_paged_batch_gives_up_cleanly():
    """The polled merge of partitions dealt out by the lengths, with a wait bound of zero: a workgroup that would have to wait gives
    up, every kernel ends, the next wait reports it, and the context goes on - with the second launch, and polled again on request."""
    announce("polled paged batch, zero wait bound")
    g = fa.Foundry(0)
    try:
        lens = [700, 30, 1000, 500, 1023, 999, 4]
        b = Batch(g, np.random.default_rng(5), 16, 2, 128, 16, lens, fa.ROPE_NEOX)
        want = [b.want(i, n)[1] for i, n in enumerate(lens)]

        def right():
            got = b.out()  # waits for the stream
            return all(max_abs(got[i], w) <= TOL for i, w in enumerate(want))

        for _ in range(4):
            g.set_decode_variant(0, 2)
            g.set_decode_poll_spin_us(0)
            b.step()
            try:
                assert right()  # nobody had to wait
            except fa.FoundryError as e:
                assert e.variant == "OperationFailed" and "waited longer" in str(e)
                b.step()
                assert right()
            g.synchronize()
        g.set_decode_poll_spin_us(5000)
        g.set_decode_variant(0, 2)
        for _ in range(3):
            b.step()
            assert right()
        assert all(b.caches_match(i) for i in range(len(lens)))
    finally:
        g.close()


@pytest.mark.usefixtures("prefill_variant")
@pytest.mark.parametrize("H,Hkv,D,bs,prefix,M", [
    (6, 2, 128, 16, 333, 100),    # context ends inside a block and inside a key tile
    (14, 2, 64, 48, 70, 37),      # block size not a power of two, head_dim 64
    (8, 8, 128, 32, 0, 129),      # no prefix, one row into a second query tile
    (4, 2, 128, 16, 2000, 32),    # a 32-row chunk after a long prefix: few query tiles, split over the keys
    (24, 8, 128, 16, 1111, 32),   # the same at the Llama-3.2-3B shape: the three heads of a KV group share an item
    (14, 2, 64, 32, 500, 9),      # nine rows, groups of seven heads
])
def test_paged_prefill_chunk_after_prefix(H, Hkv, D, bs, prefix, M):
    """A prefill chunk attending a paged cache that already holds a prefix (sequence 1 of 3, random block
    permutation), against the oracle over the gathered contiguous cache."""
    announce("paged prefill chunk", H, Hkv, D, bs, prefix, M)
    f = ctx()
    rng = np.random.default_rng(prefix * 7 + M)
    N = prefix + M
    lens = [5, N, 40]
    ks = [h16(rng.normal(size=(Hkv, n, D))) for n in lens]
    vs = [h16(rng.normal(size=(Hkv, n, D))) for n in lens]
    pg = Paged(f, rng, lens, Hkv, D, bs, extra_tokens=0)
    pg.fill_from(ks, vs)
    pg.upload()
    q = h16(rng.normal(size=(H, M, D)))
    dq, dout = f.array(q), f.zeros((M, H * D))
    f.flash_prefill_paged(dq.arg(), pg.desc, 1, dout.arg(), True, prefix, H, N, M)
    f.synchronize()
    got = dout.download()
    want = orc.sdpa_prefill(q, ks[1], vs[1], H, Hkv, D, M, N, prefix, N, causal=True, n_threads=8)  # token-major
    assert np.all(np.isfinite(got))
    assert max_abs(got, want) <= TOL
    pg.free()
    for b in (dq, dout):
        b.free()


@pytest.mark.parametrize("D,M,prefix", [(64, 200, 700), (128, 129, 448)])
def test_tiled_prefill_bits_whatever_the_pages(D, M, prefix):
    """The tiled kernel for pools with 32-bit offsets and pages of a power of two, and the one for other pages and for pools of 4 GiB:
    the bits of the contiguous cache."""
    announce("tiled prefill, pools", D, M, prefix)
    f = ctx()
    rng = np.random.default_rng(D + M)
    H, Hkv, N = 6, 2, prefix + M
    rows = [f.array(h16(rng.normal(size=(N, h * D)))) for h in (H, Hkv, Hkv)]
    q, q_rot = f.array(h16(rng.normal(size=(H, M, D)))), f.zeros((H, N, D))
    cos, sin = (f.array(t) for t in fa.rope_tables(1e4, D, N))
    lens, do = f.array(np.array([N], np.uint32)), f.zeros((M, H * D))
    ins = [r.arg() for r in rows]
    try:
        f.set_prefill_variant(2)
        f.set_prefill_split_k(1)
        kc, vc = f.empty((Hkv, N, D)), f.empty((Hkv, N, D))
        p = fa.KvPrepFusedParams.make(H, Hkv, D, N, 0, N, fa.ROPE_NEOX)
        f.kv_prep_fused(*ins, q_rot.arg(), kc.arg(), vc.arg(), cos.arg(), sin.arg(), p)
        f.flash_attention(q.arg(), kc.arg(), vc.arg(), do.arg(), True, prefix, H, D, N, M)
        want = do.download().view(np.uint16).copy()
        assert np.any(want)
        for bs, n_pages in ((16, 0), (64, 0), (48, 0), (16, 2 ** 32 // (Hkv * 16 * D * 2))):
            nb = (N + bs - 1) // bs
            n_pages = n_pages or nb + 3
            table = rng.permutation(n_pages)[:nb].astype(np.int32)
            if n_pages - 1 not in table:
                table[-1] = n_pages - 1
            kp, vp, bt = f.empty((n_pages, Hkv, bs, D)), f.empty((n_pages, Hkv, bs, D)), f.array(table)
            cache = fa.paged_kv(kp, vp, bt, lens, n_pages, Hkv, bs, D, 1, nb)
            p = fa.KvPrepFusedParams.make(H, Hkv, D, N, 0, nb * bs, fa.ROPE_NEOX)
            f.kv_prep_fused_paged(*ins, q_rot.arg(), cache, 0, cos.arg(), sin.arg(), p)
            do.upload(np.zeros((M, H * D), np.float16))
            f.flash_prefill_paged(q.arg(), cache, 0, do.arg(), True, prefix, H, N, M)
            assert np.array_equal(do.download().view(np.uint16), want), (bs, n_pages)
            for b in (kp, vp, bt):
                b.free()
    finally:
        f.set_prefill_variant(0)
        f.set_prefill_split_k()
    for b in rows + [q, q_rot, cos, sin, lens, do, kc, vc]:
        b.free()
