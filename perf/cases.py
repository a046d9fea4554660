"""What the library is timed on: the work that a program which serves a model through it has it do.

A case is one pass over one or several layers of that work - a decode step, a batch of decode steps, a prompt or a chunk of
one, the attention block around either (FusedQkv, attention, o_proj with its residual), the int8 decode session, the growth of
the KV cache - with tensors that live on the GPU, through the entry points of test-burn_amd/foundry_attn.py. The layers' shapes
are those of this repository's benchmark configurations.
"""
import math
import os
import sys
import weakref

import torch

sys.path.insert(0, os.path.abspath("test-burn_amd"))
import foundry_attn as fa  # noqa: E402

# Shapes of bench.py's configurations: query heads, KV heads, head_dim, layers, RoPE base and pairing, biases on Q/K/V, and
# every how many layers RoPE is left out (0 = never). The hidden size is heads * head_dim.
MODELS = {
    "qwen2.5-0.5b": dict(h=14, hkv=2, d=64, layers=24, theta=1e6, mode=fa.ROPE_NEOX, bias=True, nope=0),
    "qwen2.5-3b": dict(h=16, hkv=2, d=128, layers=36, theta=1e6, mode=fa.ROPE_NEOX, bias=True, nope=0),
    "llama3.2-3b": dict(h=24, hkv=8, d=128, layers=28, theta=5e5, mode=fa.ROPE_NORMAL, bias=False, nope=0),
    "smollm3": dict(h=16, hkv=4, d=128, layers=36, theta=1e6, mode=fa.ROPE_NEOX, bias=False, nope=4),
}


def listed():
    return [
        # The smallest calls there are: a layer's decode step of the small model at a short context, called eagerly.
        dict(name="decode_0.5b_1k", kind="decode", model="qwen2.5-0.5b", layers=2, ctx=1024, dtype="f16", graph=False),
        # The headline: the attention of one token through all layers at 8K context, replayed as a recorded graph.
        dict(name="decode_3b_8k_28_layers", kind="decode", model="llama3.2-3b", layers=28, ctx=8192, dtype="f16", graph=True),
        # A long document: a few layers of a bf16 cache at an odd length.
        dict(name="decode_3b_50001_bf16", kind="decode", model="llama3.2-3b", layers=2, ctx=50001, dtype="bf16", graph=False),
        # A server's decode step: 32 sequences of very different lengths in a paged cache.
        dict(name="decode_batch_32_paged", kind="batch", model="qwen2.5-3b", layers=1, seqs=32, lo=512, hi=16384, page=16, dtype="f16"),
        # One token through the attention blocks of the small model with Q8_0 weights, as the reference's own throughput
        # figures are taken: projections, decode step and o_proj of every layer, replayed as a graph.
        dict(name="block_decode_0.5b_q8", kind="block", model="qwen2.5-0.5b", layers=24, m=1, prefix=700, weights="q8",
             canonical=True, paged=False, graph=True),
        # The same for a server's batch: the tokens of 24 sequences go through Q4_0 projections together.
        dict(name="block_batch_24_q4", kind="block_batch", model="qwen2.5-3b", layers=2, seqs=24, lo=100, hi=4000, page=16,
             weights="q4", canonical=True),
        # A chunk of the reference's default size after a long prefix.
        dict(name="block_chunk32_3b_8k", kind="block", model="llama3.2-3b", layers=4, m=32, prefix=8160, weights="f16",
             canonical=True, paged=False, graph=False),
        # A prompt in one piece: the attention block is matrix products and causal attention.
        dict(name="block_prompt_3b_2048", kind="block", model="llama3.2-3b", layers=1, m=2048, prefix=0, weights="f16",
             canonical=True, paged=False, graph=False),
        # A chunk of nearly the largest size the chunk schedule uses (512), in the middle of a prompt, small model, Q8_0, paged.
        dict(name="block_chunk500_0.5b_q8", kind="block", model="qwen2.5-0.5b", layers=4, m=500, prefix=1000, weights="q8",
             canonical=True, paged=True, graph=False),
        # A long prompt's attention alone (append of its K/V rows, then causal attention), bf16, not a multiple of any tile.
        dict(name="prefill_3b_8001_bf16", kind="prefill", model="llama3.2-3b", layers=1, m=8001, prefix=0, dtype="bf16", paged=False),
        # An int8 session at 32K: the state is built from the prompt's cache, then the first tokens are decoded on it.
        dict(name="int8_smollm3_32k", kind="int8", model="smollm3", ctx=32768, steps=16),
        # The cache outgrown at 8K context: every layer's K and V move to a cache of twice the capacity.
        dict(name="growth_3b_8k", kind="growth", model="llama3.2-3b", layers=28, tokens=8448, dtype="f16"),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    model = rng.choice(sorted(MODELS))
    s = MODELS[model]
    kind = rng.choice(["decode", "batch", "prefill", "block", "block", "block_batch", "int8", "growth"])
    row = 4 * s["hkv"] * s["d"]  # bytes of one token's K and V in one layer
    c = dict(kind=kind, model=model)
    if kind == "decode":
        ctx = log_int(64, 131072)
        most = max(2, min(s["layers"], int(1.2e9 / (row * ctx))))
        graph = rng.random() < 0.5
        c.update(layers=rng.randint(2, most if graph else min(most, 4)), ctx=ctx, dtype=rng.choice(["f16", "bf16"]), graph=graph)
    elif kind == "batch":
        seqs = log_int(2, 64)
        hi = log_int(256, min(16384, int(1.2e9 / (row * seqs))))
        c.update(layers=1, seqs=seqs, lo=log_int(16, hi), hi=hi, page=rng.choice([16, 32, 64]), dtype=rng.choice(["f16", "bf16"]))
    elif kind == "prefill":
        m = log_int(16, 8000)
        c.update(layers=1, m=m, prefix=rng.choice([0, log_int(16, 16384 - 2 * m) if m < 4000 else 0]), dtype=rng.choice(["f16", "bf16"]),
                 paged=rng.random() < 0.5)
    elif kind == "block":
        m = rng.choice([1, log_int(2, 64), log_int(33, 512), log_int(64, 2048)])
        c.update(layers=rng.randint(1, max(1, min(4, 3000 // m))), m=m, prefix=log_int(16, 8192), weights=rng.choice(["f16", "q8", "q4"]),
                 canonical=rng.random() < 0.7, paged=m > 1 and rng.random() < 0.5, graph=m <= 64 and rng.random() < 0.5)
    elif kind == "block_batch":
        layers, seqs = rng.randint(1, 4), log_int(2, 64)
        hi = log_int(256, min(8192, int(1.2e9 / (row * seqs * layers))))
        c.update(layers=layers, seqs=seqs, lo=log_int(16, hi), hi=hi, page=rng.choice([16, 32]),
                 weights=rng.choice(["f16", "q8", "q4"]), canonical=rng.random() < 0.7)
    elif kind == "int8":
        c.update(ctx=log_int(256, 32768), steps=rng.randint(2, 16))
    else:
        tokens = log_int(100, 16384)
        most = max(1, min(s["layers"], int(9e8 / (row * tokens))))
        c.update(layers=rng.randint(1, most), tokens=tokens, dtype=rng.choice(["f16", "bf16"]))
    return c


def lengths(case):
    """The tokens each sequence of a batch already holds: spread evenly over [lo, hi], in no order."""
    n, lo, hi = case["seqs"], case["lo"], case["hi"]
    return [lo + int((hi - lo) * ((0.5 + i * 0.6180339887498949) % 1.0)) for i in range(n)]


def work(case):
    s, kind = MODELS[case["model"]], case["kind"]
    h, hkv, d = s["h"], s["hkv"], s["d"]
    dm, kvd = h * d, hkv * d
    layers, m, pairs, rows = case.get("layers", 1), case.get("m", 1), 0, 0
    if kind == "growth":
        return {"bytes": 2 * 4 * kvd * layers * case["tokens"], "flops": 0}
    if kind == "int8":
        n, steps = case["ctx"], case["steps"]
        build = 2 * kvd * n + kvd * n + 2 * hkv * n / 32  # f16 K in, int8 K and scales out
        step = (3 * kvd + 2 * hkv / 32) * (n + steps / 2) + 4 * kvd + 4 * dm
        return {"bytes": build + steps * step, "flops": 2 * kvd * n + steps * 4 * dm * (n + steps / 2)}
    if kind in ("batch", "block_batch"):
        m = case["seqs"]
        rows = pairs = sum(lengths(case)) + m
    elif kind == "decode":
        rows = pairs = case["ctx"] + 1
    else:
        p = case["prefix"]
        rows, pairs = p + m, m * p + m * (m + 1) // 2
    # K and V rows read or written once, the new tokens' q, k, v read and the attention's output written
    nbytes, flops = 4 * kvd * rows, 4 * dm * pairs
    if kind in ("block", "block_batch"):
        n = 2 * dm + 2 * kvd  # weight rows of Q, K, V and o_proj
        per = {"f16": 2.0, "q8": 1.0 + 2 / 32, "q4": 0.5 + 2 / 32}[case["weights"]]
        nbytes += n * dm * per + 4 * m * dm  # hidden in and out; q, k, v and the attention's output need not leave the chip
        flops += 2 * m * n * dm
    else:
        nbytes += 2 * m * (2 * dm + 2 * kvd)
    return {"bytes": layers * nbytes, "flops": layers * flops}


def tolerance(case):
    if case["kind"] == "growth":
        return "exact"
    if case["kind"] == "int8":  # int8 codes: another order of the mean's sum can move a value across a rounding boundary
        return {"rel": 4e-3, "differ": 1e-3}
    if case.get("dtype") == "bf16":
        return {"rel": 1e-2}
    # f16 at every step, and in a block each layer's rounding is the next one's input
    return {"rel": 2e-3 * math.sqrt(case["layers"] if case["kind"].startswith("block") else 1)}


# ---------------------------------------------------------------------------------------------------------------- preparing

_ctx = []
_DTYPES = {torch.float16: fa.DTYPE_F16, torch.bfloat16: fa.DTYPE_BF16, torch.float32: fa.DTYPE_F32, torch.int8: fa.DTYPE_I8,
           torch.uint8: fa.DTYPE_U8, torch.int32: fa.DTYPE_I32}


def context():
    """One context for the whole program: its launches share the GPU in one stream's order."""
    if not _ctx:
        _ctx.append(fa.Foundry(0))
    return _ctx[0]


def targ(t, dims=None, dtype=None):
    """The library's tensor argument for a contiguous torch tensor (or for its bytes, as dims of dtype)."""
    a = fa.TensorArg()
    a.buffer, a.offset = t.data_ptr(), 0
    a.dtype = _DTYPES[t.dtype] if dtype is None else dtype
    dims = tuple(t.shape) if dims is None else dims
    a.rank = len(dims)
    stride = 1
    for i in reversed(range(len(dims))):
        a.dims[i], a.strides[i] = dims[i], stride
        stride *= dims[i]
    return a


class Ptr:
    """What the binding's calls that take a buffer want: an object with the device address."""

    def __init__(self, t):
        self.ptr = t.data_ptr()


class State:
    """Tensors, arguments and, where the program records one, the graph of a pass."""

    def __init__(self, case, seed):
        self.case, self.s, self.f = case, MODELS[case["model"]], context()
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.dt = torch.bfloat16 if case.get("dtype") == "bf16" else torch.float16
        self.keep, self.graph, self.pos, self.bound = [], None, None, 0

    def normal(self, *shape, scale=1.0, dtype=None):
        t = torch.randn(shape, generator=self.gen, device="cuda", dtype=dtype or self.dt)
        if scale != 1.0:
            t *= scale
        self.keep.append(t)
        return t

    def zeros(self, *shape, dtype=None):
        t = torch.zeros(shape, device="cuda", dtype=dtype or self.dt)
        self.keep.append(t)
        return t

    def tables(self, rows):
        t = [torch.from_numpy(x).cuda() for x in _tables(self.s["theta"], self.s["d"], rows)]
        self.keep += t
        self.cos, self.sin = targ(t[0]), targ(t[1])

    def params(self, layer, seq_len, position, capacity):
        s = self.s
        return fa.KvPrepFusedParams.make(s["h"], s["hkv"], s["d"], seq_len, position, capacity, s["mode"], layer, s["nope"])

    def position(self, pos, capacity):
        """A recorded step reads its position from device memory, so that the program can replay it at the next one."""
        t = torch.tensor([pos], device="cuda", dtype=torch.int32)
        self.keep.append(t)
        self.pos, self.bound = Ptr(t), capacity

    def record(self, enqueue):
        """Runs the pass once (scratch memory grows outside a capture) and records it."""
        torch.cuda.synchronize()
        enqueue(self)
        self.f.synchronize()
        self.f.start_capture()
        enqueue(self)
        self.graph = self.f.end_capture()
        weakref.finalize(self, self.graph.destroy)


_table_cache = {}


def _tables(theta, d, rows):
    rows = (rows + 4095) // 4096 * 4096
    key = (theta, d)
    if key not in _table_cache or _table_cache[key][0].shape[0] < rows:
        _table_cache[key] = fa.rope_tables(theta, d, rows)
    return [x[:rows] for x in _table_cache[key]]


def paged_cache(st, layers, seqs, tokens, page):
    """Pools of all layers, filled; each sequence's blocks lie anywhere in them. Returns (K, V, one PagedKv per layer, lengths)."""
    s = st.s
    per_seq = (max(tokens) + 1 + page - 1) // page
    n_blocks = seqs * per_seq
    k, v = (st.normal(layers, n_blocks, s["hkv"], page, s["d"]) for _ in range(2))
    table = torch.randperm(n_blocks, generator=st.gen, device="cuda").to(torch.int32).reshape(seqs, per_seq).contiguous()
    lens = torch.tensor(tokens, device="cuda", dtype=torch.int32)
    st.keep += [table, lens]
    caches = [fa.paged_kv(Ptr(k[i]), Ptr(v[i]), Ptr(table), Ptr(lens), n_blocks, s["hkv"], page, s["d"], seqs, per_seq)
              for i in range(layers)]
    return k, v, caches, lens


def matrix(st, rows, k, weights, canonical):
    """One projection's weights, of unit gain, and its block scales: (weights, scales or None) as tensor arguments."""
    if weights == "f16":
        return targ(st.normal(rows, k, scale=k ** -0.5, dtype=torch.float16)), None
    scales = torch.rand(rows, k // 32, generator=st.gen, device="cuda") * 0.5 + 0.75
    if weights == "q8":
        w = (torch.randn(rows, k, generator=st.gen, device="cuda") * 36).round_().clamp_(-127, 127).to(torch.int8)
        scales = (scales * k ** -0.5 / 36).half()
        arg = targ(w, dtype=fa.DTYPE_Q8_0)
    else:
        w = torch.randint(0, 256, (rows, k // 2), generator=st.gen, device="cuda", dtype=torch.uint8)
        scales = (scales * k ** -0.5 / 4.6).half()
        arg = targ(w, dims=(rows, k), dtype=fa.DTYPE_Q4_0)
    st.keep += [w, scales]
    return arg, targ(scales)


def projections(st, case, layers, m):
    """FusedQkv's and o_proj's operands of every layer and the hidden states between them."""
    s = st.s
    dm, kvd = s["h"] * s["d"], s["hkv"] * s["d"]
    st.hidden = st.normal(layers + 1, m, dm, dtype=torch.float16)
    st.attn = st.zeros(layers, m, dm)
    st.q_rot = st.zeros(s["h"], m, s["d"])
    st.qkv = [targ(st.zeros(m, n)) for n in (dm, kvd, kvd)]
    st.layers = []
    for i in range(layers):
        w = [matrix(st, n, dm, case["weights"], case["canonical"]) for n in (dm, kvd, kvd, dm)]
        gamma = st.normal(dm, scale=0.1, dtype=torch.float16).add_(1.0)
        biases = tuple(targ(st.normal(n, scale=0.5, dtype=torch.float16)) for n in (dm, kvd, kvd)) if s["bias"] else None
        quant = case["weights"] != "f16"
        st.layers.append(dict(w=[x[0] for x in w[:3]], scales=tuple(x[1] for x in w[:3]) if quant else None, w_o=w[3][0], s_o=w[3][1],
                              gamma=targ(gamma), biases=biases, x=targ(st.hidden[i]), y=targ(st.hidden[i + 1]),
                              attn=targ(st.attn[i])))
    st.layout = fa.WEIGHT_LAYOUT_CANONICAL if case["canonical"] else fa.WEIGHT_LAYOUT_ROW_MAJOR


def prepare(case, seed):
    st = State(case, seed)
    s, kind = st.s, case["kind"]
    h, hkv, d = s["h"], s["hkv"], s["d"]
    dm, kvd = h * d, hkv * d
    layers, m = case.get("layers", 1), case.get("m", 1)
    enqueue = PASSES[kind]
    if kind == "decode":
        cap = fa.align_capacity(case["ctx"] + 1)
        st.tables(cap)
        k, v = (st.normal(layers, hkv, cap, d) for _ in range(2))
        out = st.zeros(layers, dm)
        qkv = [st.normal(layers, n) for n in (dm, kvd, kvd)]
        st.calls = [dict(q=targ(qkv[0][i:i + 1]), k=targ(qkv[1][i:i + 1]), v=targ(qkv[2][i:i + 1]), kc=targ(k[i]), vc=targ(v[i]),
                         out=targ(out[i:i + 1]), p=st.params(i, 1, case["ctx"], cap)) for i in range(layers)]
        st.out = dict(out=out, k=k, v=v)
    elif kind == "batch":
        tokens = lengths(case)
        st.tables(max(tokens) + 1)
        k, v, caches, lens = paged_cache(st, layers, case["seqs"], tokens, case["page"])
        n = case["seqs"]
        out = st.zeros(layers, n, dm)
        qkv = [st.normal(layers, n, w) for w in (dm, kvd, kvd)]
        st.bound = max(tokens) + 1
        st.calls = [dict(q=targ(qkv[0][i]), k=targ(qkv[1][i]), v=targ(qkv[2][i]), cache=caches[i], out=targ(out[i]),
                         p=st.params(i, n, 0, 0)) for i in range(layers)]
        st.out = dict(out=out, k=k, v=v)
    elif kind == "prefill":
        n = case["prefix"] + m
        st.tables(n)
        out, q_rot = st.zeros(layers, m, dm), st.zeros(h, m, d)
        qkv = [st.normal(layers, m, w) for w in (dm, kvd, kvd)]
        st.q_rot = targ(q_rot)
        if case["paged"]:
            k, v, caches, _ = paged_cache(st, layers, 1, [n], 16)
            kv = [dict(cache=c) for c in caches]
        else:
            cap = fa.align_capacity(n)
            k, v = (st.normal(layers, hkv, cap, d) for _ in range(2))
            kv = [dict(kc=targ(k[i]), vc=targ(v[i])) for i in range(layers)]
        cap = 0 if case["paged"] else cap
        st.calls = [dict(q=targ(qkv[0][i]), k=targ(qkv[1][i]), v=targ(qkv[2][i]), out=targ(out[i]),
                         p=st.params(i, m, case["prefix"], cap), **kv[i]) for i in range(layers)]
        st.out = dict(out=out, q_rot=q_rot, k=k, v=v)
    elif kind == "block":
        n = case["prefix"] + m
        st.tables(n)
        projections(st, case, layers, m)
        if case["paged"]:
            k, v, caches, _ = paged_cache(st, layers, 1, [n], 16)
            kv, cap = [dict(cache=c) for c in caches], 0
        else:
            cap = fa.align_capacity(n)
            k, v = (st.normal(layers, hkv, cap, d) for _ in range(2))
            kv = [dict(kc=targ(k[i]), vc=targ(v[i])) for i in range(layers)]
        for i, l in enumerate(st.layers):
            l.update(p=st.params(i, m, case["prefix"], cap), **kv[i])
        st.q_rot_arg = targ(st.q_rot)
        st.out = dict(hidden=st.hidden, attn=st.attn, k=k, v=v)
    elif kind == "block_batch":
        tokens = lengths(case)
        n = case["seqs"]
        st.tables(max(tokens) + 1)
        projections(st, case, layers, n)
        k, v, caches, lens = paged_cache(st, layers, n, tokens, case["page"])
        st.bound = max(tokens) + 1
        for i, l in enumerate(st.layers):
            l.update(p=st.params(i, n, 0, 0), cache=caches[i])
        st.out = dict(hidden=st.hidden, attn=st.attn, k=k, v=v)
    elif kind == "int8":
        n, steps = case["ctx"], case["steps"]
        cap = fa.align_capacity(n + steps)
        st.tables(cap)

        def outliers(*shape):  # 1 % of the values at eight standard deviations
            t = st.normal(*shape)
            t[torch.rand(shape, generator=st.gen, device="cuda") < 0.01] *= 8
            return t

        k_f16, v = outliers(hkv, cap, d), outliers(hkv, cap, d)
        q, k_new, v_new = st.normal(steps, dm), st.normal(steps, kvd), st.normal(steps, kvd)
        out = st.zeros(steps, dm)
        bufs = dict(k_q=st.zeros(hkv, cap, d, dtype=torch.int8), k_scale=st.zeros(hkv, (cap + 31) // 32),
                    k_tail=st.zeros(hkv, 32, d), v=v, q_q=st.zeros(h, d, dtype=torch.int8),
                    k_mean=st.zeros(hkv, d, dtype=torch.float32), q_scale=st.zeros(h, dtype=torch.float32))
        st.cache = fa.SageCache(*[bufs[x].data_ptr() for x in ("k_q", "k_scale", "k_tail", "v", "q_q", "k_mean", "q_scale")],
                                h, hkv, cap, d)
        st.k_f16 = Ptr(k_f16)
        st.calls = [dict(q=targ(q[i:i + 1]), k=targ(k_new[i:i + 1]), v=targ(v_new[i:i + 1]), out=targ(out[i:i + 1]),
                         p=st.params(0, 1, n + i, cap)) for i in range(steps)]
        st.out = dict(out=out, **bufs)
    else:
        tokens = case["tokens"]
        old = fa.align_capacity(tokens)
        new = fa.grown_capacity(old, old + 1, 1 << 20)
        src, dst = st.normal(2 * layers, hkv, old, d), st.zeros(2 * layers, hkv, new, d)
        st.src, st.dst = [targ(src[i]) for i in range(2 * layers)], [targ(dst[i]) for i in range(2 * layers)]
        st.out = dict(kv=dst)
    if case.get("graph"):
        if m == 1:
            st.position(case["ctx"] if kind == "decode" else case["prefix"], cap)
        st.record(enqueue)
    torch.cuda.synchronize()
    return st


# ------------------------------------------------------------------------------------------------------------------ running

def _decode(st):
    for c in st.calls:
        st.f.decode_step_fused(c["q"], c["k"], c["v"], None, c["kc"], c["vc"], st.cos, st.sin, c["out"], c["p"], st.pos, st.bound)


def _batch(st):
    for c in st.calls:
        st.f.decode_step_fused_paged(c["q"], c["k"], c["v"], None, c["cache"], st.cos, st.sin, c["out"], c["p"], st.bound)


def _attend(st, c, q_rot, out, m, prefix):
    s, n = st.s, prefix + m
    if "cache" in c:
        st.f.flash_prefill_paged(q_rot, c["cache"], 0, out, True, prefix, s["h"], n, m)
    else:
        st.f.flash_attention(q_rot, c["kc"], c["vc"], out, True, prefix, s["h"], s["d"], n, m)


def _prefill(st):
    m, prefix = st.case["m"], st.case["prefix"]
    for c in st.calls:
        if "cache" in c:
            st.f.kv_prep_fused_paged(c["q"], c["k"], c["v"], st.q_rot, c["cache"], 0, st.cos, st.sin, c["p"])
        else:
            st.f.kv_prep_fused(c["q"], c["k"], c["v"], st.q_rot, c["kc"], c["vc"], st.cos, st.sin, c["p"])
        _attend(st, c, st.q_rot, c["out"], m, prefix)


def _fused_qkv(st, l, m):
    s = st.s
    dm, kvd = s["h"] * s["d"], s["hkv"] * s["d"]
    st.f.fused_qkv(l["x"], *l["w"], *st.qkv, dm, dm, kvd, m=m, gamma=l["gamma"], biases=l["biases"], layout=st.layout, scales=l["scales"])


def _o_proj(st, l, m):
    dm = st.s["h"] * st.s["d"]
    st.f.matmul(l["attn"], l["w_o"], l["y"], m, dm, dm, c=l["x"], transpose_b=not st.case["canonical"], beta=1.0, b_scales=l["s_o"])


def _block(st):
    m, prefix = st.case["m"], st.case["prefix"]
    for l in st.layers:
        if m == 1:
            _fused_qkv(st, l, 1)
            st.f.decode_step_fused(*st.qkv, None, l["kc"], l["vc"], st.cos, st.sin, l["attn"], l["p"], st.pos, st.bound)
        else:
            where = dict(paged=l["cache"]) if "cache" in l else dict(k_cache=l["kc"], v_cache=l["vc"])
            st.f.fused_qkv_kv_prep(l["x"], *l["w"], st.s["h"] * st.s["d"], st.q_rot_arg, st.cos, st.sin, l["p"], gamma=l["gamma"],
                                   biases=l["biases"], layout=st.layout, scales=l["scales"], **where)
            _attend(st, l, st.q_rot_arg, l["attn"], m, prefix)
        _o_proj(st, l, m)


def _block_batch(st):
    n = st.case["seqs"]
    for l in st.layers:
        _fused_qkv(st, l, n)
        st.f.decode_step_fused_paged(*st.qkv, None, l["cache"], st.cos, st.sin, l["attn"], l["p"], st.bound)
        _o_proj(st, l, n)


def _int8(st):
    st.f.sage_cache_build(st.k_f16, st.case["ctx"], st.cache)
    for c in st.calls:
        st.f.sage_decode_step(c["q"], c["k"], c["v"], st.cache, st.cos, st.sin, c["out"], c["p"])


def _growth(st):
    st.f.kv_prefix_copy_batch(st.src, st.dst, st.case["tokens"])


PASSES = dict(decode=_decode, batch=_batch, prefill=_prefill, block=_block, block_batch=_block_batch, int8=_int8, growth=_growth)


def run(st):
    if st.graph is not None:
        st.graph.launch()
    else:
        PASSES[st.case["kind"]](st)
    return st.out
