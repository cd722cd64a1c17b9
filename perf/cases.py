"""Workloads of the attention, RoPE-append and MatVec entry points for timing and comparing builds.

Every case is work that an engine on this library has it do for one layer (or a few), through
the package's public calls on device tensors: decode attention over a paged cache, a prompt
chunk or a speculative verify (append, then causal attention), a captured decode step of an
attention block, MLA absorbed attention with and without its projections, and the MatVecs of a
layer.  Sizes are those of bench.py and the tests (a tiny GQA shape, the 8B and 70B GQA shapes,
the 128-head 512 + 64 MLA shape) and generic ones around them.

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs, caches and weights of one pass, on the GPU
    run(state)          one pass; returns its outputs
    work(case)          bytes and flops a pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   the outputs in 64-bit arithmetic by plain torch
"""
import math

import torch

import qauntrunner_amd as qr

THETA = 500000.0
PAGE = 256
CODE = {"F32": 0, "F16": 1, "BF16": 2, "Q4_0": 3, "Q8_0": 4, "Q4_K": 6, "Q6_K": 7}
BLOCK = {"F32": (1, 4), "F16": (1, 2), "BF16": (1, 2), "Q4_0": (32, 20), "Q8_0": (32, 34), "Q4_K": (256, 144),
         "Q6_K": (256, 210)}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # the smallest call: a tiny model's layer, where the launch and the host path count
        dict(name="decode-tiny-f32", kind="decode", heads=8, kv=2, D=64, B=1, lo=512, hi=512, dtype="f32"),
        # one token of an 8B-shape layer at the end of a long context, in the default cache type
        dict(name="decode-8b-f32-32k", kind="decode", heads=32, kv=8, D=128, B=1, lo=32768, hi=32768, dtype="f32"),
        # a serving batch: sequences of very different lengths decode together
        dict(name="decode-batch-bf16", kind="decode", heads=32, kv=8, D=128, B=16, lo=130, hi=16000, dtype="bf16"),
        # a serving loop's captured token step: QKV MatVecs, RoPE + append, attention, output
        # MatVec of four layers at an ordinary context length
        dict(name="step-8b-q4k", kind="step", heads=32, kv=8, D=128, layers=4, pos=1500, max_seq=4096, wfmt="Q4_K",
             dtype="f16"),
        # a chunk of a long prompt with 16-bit queries, as an engine with bf16 activations has them
        dict(name="prefill-8b-bf16", kind="chunk", heads=32, kv=8, D=128, pos0=6144, nq=2048, dtype="bf16", rope=False,
             q_dtype="bf16"),
        # a chunk of a prompt in the default cache type, RoPE included
        dict(name="prefill-8b-f32", kind="chunk", heads=32, kv=8, D=128, pos0=1536, nq=512, dtype="f32", rope=True,
             q_dtype="f32"),
        # a whole short prompt of an odd length
        dict(name="prefill-short-f16", kind="chunk", heads=32, kv=8, D=128, pos0=0, nq=333, dtype="f16", rope=True,
             q_dtype="f32"),
        # speculative verify: eight drafts at the end of a very long context, 70B shape
        dict(name="verify-70b-f16", kind="chunk", heads=64, kv=8, D=128, pos0=131072, nq=8, dtype="f16", rope=True,
             q_dtype="f32"),
        # MLA absorbed attention in the default latent type
        dict(name="mla-f32", kind="mla", heads=128, lora=512, rope_dim=64, n=4096, dtype="f32"),
        # an MLA layer's whole absorbed block for one token, 16-bit latents, quantized projections
        dict(name="mla-layer-q8", kind="mla_layer", heads=128, lora=512, rope_dim=64, nope=128, vdim=128, n=16384,
             dtype="bf16", wfmt="Q8_0"),
        # every MatVec of an 8B-shape layer for one token
        dict(name="matvec-8b-q4k", kind="matvec", dim=4096, kvdim=1024, ffn=14336, wfmt="Q4_K", nq=1),
        # the same for the eight drafts of a verify
        dict(name="matvec-8b-q8-n8", kind="matvec", dim=4096, kvdim=1024, ffn=14336, wfmt="Q8_0", nq=8),
    ]


# ------------------------------------------------------------------ drawn cases
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


GQA = [(8, 2), (16, 16), (24, 8), (28, 4), (32, 8), (64, 8)]


def _gqa(rng):
    heads, kv = rng.choice(GQA)
    return heads, kv, rng.choice([64, 128, 128, 128, 96, 256])


def draw(rng):
    """A case of the ranges of listed(); within a kind none costs more than its listed cases."""
    kind = rng.choice(["decode", "step", "chunk", "mla", "mla_layer", "matvec"])
    dtype = rng.choice(["f32", "f16", "bf16"])
    while True:
        if kind == "decode":
            heads, kv, D = _gqa(rng)
            hi = _log(rng, 40, 40000)
            c = dict(kind=kind, heads=heads, kv=kv, D=D, B=_log(rng, 1, 32), lo=max(1, hi // rng.choice([1, 2, 40])),
                     hi=hi, dtype=dtype)
        elif kind == "step":
            heads, kv, D = rng.choice([(8, 2, 64), (16, 4, 128), (32, 8, 128), (16, 16, 64), (28, 4, 128)])
            pos = _log(rng, 20, 6000)
            c = dict(kind=kind, heads=heads, kv=kv, D=D, layers=rng.choice([2, 3, 4]), pos=pos,
                     max_seq=pos + rng.choice([1, 500, 2500]), wfmt=rng.choice(["Q4_K", "Q8_0", "F16", "BF16"]),
                     dtype=dtype)
        elif kind == "chunk":
            heads, kv, D = _gqa(rng)
            rope = rng.random() < 0.7
            c = dict(kind=kind, heads=heads, kv=kv, D=D, pos0=rng.choice([0, _log(rng, 10, 60000)]),
                     nq=_log(rng, 2, 2048), dtype=dtype, rope=rope,
                     q_dtype="f32" if rope or rng.random() < 0.3 else dtype)
        elif kind == "mla":
            lora, rope_dim = rng.choice([(512, 64), (512, 64), (512, 64), (256, 32)])
            c = dict(kind=kind, heads=rng.choice([16, 20, 64, 128]), lora=lora, rope_dim=rope_dim,
                     n=_log(rng, 50, 16384), dtype=dtype)
        elif kind == "mla_layer":
            c = dict(kind=kind, heads=rng.choice([16, 20, 64, 128]), lora=512, rope_dim=64, nope=128, vdim=128,
                     n=_log(rng, 50, 16384), dtype=dtype, wfmt=rng.choice(["F32", "F16", "BF16", "Q8_0", "Q4_0", "Q4_K", "Q6_K"]))
        else:
            dim, kvdim, ffn = rng.choice([(1024, 256, 2816), (2048, 512, 5632), (3072, 1024, 8192), (4096, 1024, 14336)])
            c = dict(kind=kind, dim=dim, kvdim=kvdim, ffn=ffn, wfmt=rng.choice(list(CODE)), nq=rng.choice([1, _log(rng, 2, 48)]))
        if _cost(c) <= _most(c):
            return c


def _plain(c):
    """Attention outside the 16-bit tile shapes (fp32, other head sizes and groups): more time per flop."""
    if c["kind"] == "chunk":
        g = c["heads"] // c["kv"]
        return c["dtype"] == "f32" or c["D"] not in (64, 128) or g & (g - 1) != 0
    return c["kind"] in ("mla", "mla_layer") and (c["dtype"] == "f32" or c["lora"] != 512)


def _cost(c):
    """Rough units of work for bounding a drawn case."""
    w = work(c)
    if _plain(c):
        return w["flops"] + 100 * w["bytes"]
    return max(100 * w["bytes"], w["flops"])


def _most(c):
    """The largest listed case of the kind (for MLA of either kind; a plain one for a plain one)."""
    kind = c["kind"][:3]
    return max(_cost(l) for l in listed() if l["kind"][:3] == kind and _plain(l) == _plain(c))


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _rows(g, n, width, dtype):
    """n rows of N(0,1) cache values in the cache's type, made in pieces."""
    out = torch.empty(n, width, dtype=TORCH[dtype], device="cuda")
    for i in range(0, n, 16384):
        out[i:i + 16384] = _randn(g, min(16384, n - i), width)
    return out


def _bits(x):
    return x if x.dtype == torch.float32 else x.view(torch.int16)


def lengths(c):
    """Cached tokens of each sequence of a batch: spread over lo..hi by their logarithm, not sorted."""
    B = c["B"]
    order = [(i * 7 + 3) % B if math.gcd(7, B) == 1 else i for i in range(B)]
    return [max(1, int(round(c["lo"] * (c["hi"] / c["lo"]) ** ((i + 1) / B)))) for i in order]


def _weights(g, fmt, rows, cols):
    """rows x cols weights of format fmt as raw bytes: N(0, 0.05^2) for the float formats, random
    quants under scales that vary from block to block for the others."""
    if fmt in ("F32", "F16", "BF16"):
        t = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[fmt]
        return (_randn(g, rows, cols) * 0.05).to(t).view(torch.uint8).reshape(-1)
    bs, bb = BLOCK[fmt]
    nb = rows * cols // bs
    raw = torch.randint(0, 256, (nb, bb), dtype=torch.uint8, device="cuda", generator=g)

    def scale(at, mean):
        d = mean * (0.5 + torch.rand(nb, device="cuda", generator=g))
        raw[:, at:at + 2] = d.half().view(torch.uint8).view(nb, 2)
    if fmt == "Q8_0":
        scale(0, 0.05 / 127)
    elif fmt == "Q4_0":
        scale(0, 0.05 / 8)
        raw[:, 18:] = 0
    elif fmt == "Q4_K":
        scale(0, 0.05 / 15 / 32)
        scale(2, 0.05 / 63)
    else:
        scale(208, 0.05 / 32 / 64)
    return raw.reshape(-1)


def _decode(fmt, raw, rows, cols):
    """The weights of raw bytes in 64 bits (the block layouts of Dtypes.cs and BlockDequantizer.cs)."""
    if fmt in ("F32", "F16", "BF16"):
        t = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[fmt]
        return raw.view(t).view(rows, cols).double()
    bs, bb = BLOCK[fmt]
    b = raw.view(-1, bb)

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()
    if fmt == "Q8_0":
        w = half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "Q4_0":
        q = b[:, 2:18]
        w = half(0) * (torch.cat([q & 15, q >> 4], 1).double() - 8)
    elif fmt == "Q4_K":
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].reshape(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        w = (half(0) * sc)[:, :, None] * q - (half(2) * mn)[:, :, None]
    else:
        ql = b[:, 0:128].reshape(-1, 2, 2, 32).int()               # half, m & 1, l
        qh = b[:, 128:192].reshape(-1, 2, 1, 32).int()
        lo = torch.stack([ql & 15, ql >> 4], 2).reshape(-1, 2, 4, 32)  # half, m = 2 (m / 2) + (m & 1), l
        sh = torch.tensor([0, 2, 4, 6], device=raw.device).view(1, 1, 4, 1)
        q = (lo | (((qh >> sh) & 3) << 4)).double() - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(-1, 2, 4, 2)
        w = half(208)[:, :, None, None] * sc.repeat_interleave(16, 3) * q
    return w.reshape(rows, cols)


def _mats(c):
    """(rows, cols) of wq, wk, wv, wo, gate, up, down."""
    d, k, f = c["dim"], c["kvdim"], c["ffn"]
    return [(d, d), (k, d), (k, d), (d, d), (f, d), (f, d), (d, f)]


GROUPS = [[0, 1, 2], [3], [4, 5], [6]]  # MatVecs of one input run as one grouped call


def _inputs(c, seed):
    """The tensors of a case, made from the seed alone."""
    g = _gen(seed)
    k = c["kind"]
    if k == "decode":
        n = sum(lengths(c))
        return dict(K=_rows(g, n, c["kv"] * c["D"], c["dtype"]), V=_rows(g, n, c["kv"] * c["D"], c["dtype"]),
                    q=_randn(g, c["B"], c["heads"] * c["D"]) * 1.5)
    if k == "step":
        kvd, hd, L = c["kv"] * c["D"], c["heads"] * c["D"], c["layers"]
        dim = _step_dim(c)
        s = 0.05 * math.sqrt(dim)
        return dict(K=[_rows(g, c["pos"], kvd, c["dtype"]) for _ in range(L)],
                    V=[_rows(g, c["pos"], kvd, c["dtype"]) for _ in range(L)],
                    x=[_randn(g, dim) * (1.5 / s) for _ in range(L)],
                    w=[[_weights(g, c["wfmt"], r, m) for r, m in ((hd, dim), (kvd, dim), (kvd, dim), (dim, hd))]
                       for _ in range(L)])
    if k == "chunk":
        kvd, hd = c["kv"] * c["D"], c["heads"] * c["D"]
        src = "f32" if c["rope"] else c["dtype"]
        return dict(K0=_rows(g, c["pos0"], kvd, c["dtype"]), V0=_rows(g, c["pos0"], kvd, c["dtype"]),
                    K=_rows(g, c["nq"], kvd, src), V=_rows(g, c["nq"], kvd, src),
                    q=(_randn(g, c["nq"], hd) * 1.5).to(TORCH[c["q_dtype"]]))
    if k in ("mla", "mla_layer"):
        width = c["lora"] + c["rope_dim"]
        d = dict(rows=_rows(g, c["n"], width, c["dtype"]))
        if k == "mla":
            d.update(qt=_randn(g, c["heads"], c["lora"]), qrp=_randn(g, c["heads"], c["rope_dim"]))
        else:
            d.update(w=_weights(g, c["wfmt"], c["heads"] * (c["nope"] + c["vdim"]), c["lora"]),
                     q=_randn(g, c["heads"], c["nope"] + c["rope_dim"]))
        return d
    mats = _mats(c)
    return dict(w=[_weights(g, c["wfmt"], r, m) for r, m in mats],
                x=[_randn(g, c["nq"], mats[grp[0]][1]) for grp in GROUPS])


def _step_dim(c):
    """Model width of a captured step: a whole number of 256-weight blocks."""
    return -(-c["heads"] * c["D"] // 256) * 256


class _State:
    """What a program keeps between calls; the graph goes before the buffers it uses."""

    def __init__(self, **kw):
        self.graph = None
        self.__dict__.update(kw)

    def __del__(self):
        self.graph = None


def prepare(case, seed):
    c, d = case, _inputs(case, seed)
    k = c["kind"]
    if k == "decode":
        ns = lengths(c)
        kv = qr.PagedKvCache(1, c["heads"], c["kv"], c["D"], max(ns), kv_dtype=c["dtype"], max_batch=c["B"])
        kv.Reserve(sum(-(-n // PAGE) for n in ns))
        at = 0
        for s, n in enumerate(ns):
            kv.AppendRangeDev(0, 0, _bits(d["K"][at:at + n]), _bits(d["V"][at:at + n]), src_dtype=c["dtype"], seq_id=s)
            at += n
        torch.cuda.synchronize()
        return _State(kind=k, kv=kv, ids=list(range(c["B"])), pos=[n - 1 for n in ns], q=d["q"],
                      out=torch.empty_like(d["q"]), scale=1.0 / math.sqrt(c["D"]))
    if k == "step":
        L, kvd, hd = c["layers"], c["kv"] * c["D"], c["heads"] * c["D"]
        dim, scale = _step_dim(c), 1.0 / math.sqrt(c["D"])
        kv = qr.PagedKvCache(L, c["heads"], c["kv"], c["D"], c["max_seq"], kv_dtype=c["dtype"])
        kv.Reserve(L * -(-c["max_seq"] // PAGE))
        for l in range(L):
            kv.AppendRangeDev(l, 0, _bits(d["K"][l]), _bits(d["V"][l]), src_dtype=c["dtype"])
        pos = torch.full((1,), c["pos"], dtype=torch.int32, device="cuda")
        code = CODE[c["wfmt"]]
        q, kr, vr, a = (torch.empty(w, device="cuda") for w in (hd, kvd, kvd, hd))
        out = [torch.empty(dim, device="cuda") for _ in range(L)]

        def step():
            for l in range(L):
                w = d["w"][l]
                qr.matvec_group_dev(w[:3], code, [hd, kvd, kvd], dim, d["x"][l], [q, kr, vr])
                kv.AppendRopeStepDev(l, pos, q, kr, vr, THETA)
                kv.AttentionStepDev(l, [0], pos, q, a, scale)
                qr.matvec_dev(w[3], code, dim, hd, a, out[l])
        step()  # the first device-position call of a cache runs outside capture
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step()
        return _State(kind=k, kv=kv, graph=graph, out=out, keep=(d, pos, q, kr, vr, a))
    if k == "chunk":
        total = c["pos0"] + c["nq"]
        kv = qr.PagedKvCache(1, c["heads"], c["kv"], c["D"], total, kv_dtype=c["dtype"])
        kv.Reserve(-(-total // PAGE))
        if c["pos0"]:
            kv.AppendRangeDev(0, 0, _bits(d["K0"]), _bits(d["V0"]), src_dtype=c["dtype"])
        torch.cuda.synchronize()
        q = d["q"] if c["q_dtype"] == "f32" else _bits(d["q"])
        return _State(kind=k, kv=kv, c=dict(c), K=_bits(d["K"]), V=_bits(d["V"]), q=q, qr=torch.empty_like(q),
                      out=torch.empty(q.shape, device="cuda"), scale=1.0 / math.sqrt(c["D"]))
    if k in ("mla", "mla_layer"):
        m = qr.MlaLatentCache(1, c["lora"] + c["rope_dim"], c["n"], dtype=c["dtype"], rope=c["rope_dim"])
        m.Reserve(-(-c["n"] // PAGE))
        m.AppendRangeDev(0, 0, _bits(d["rows"]), src_dtype=c["dtype"])
        torch.cuda.synchronize()
        if k == "mla":
            return _State(kind=k, m=m, pos=c["n"] - 1, qt=d["qt"], qrp=d["qrp"], out=torch.empty_like(d["qt"]),
                          scale=1.0 / math.sqrt(192.0))
        return _State(kind=k, m=m, pos=c["n"] - 1, c=dict(c), q=d["q"], w=d["w"],
                      out=torch.empty(c["heads"], c["vdim"], device="cuda"))
    mats = _mats(c)
    return _State(kind=k, code=CODE[c["wfmt"]], mats=mats, w=d["w"], x=d["x"],
                  out=[torch.empty(c["nq"], r, device="cuda") for r, _ in mats])


def run(s):
    if s.kind == "decode":
        s.kv.AttentionDev(0, s.ids, s.pos, s.q, s.out, s.scale)
        return s.out
    if s.kind == "step":
        s.graph.replay()
        return s.out
    if s.kind == "chunk":
        c, q = s.c, s.q
        if c["rope"]:
            # the projection's fresh q rows; RoPE rotates them in place
            q = s.qr.copy_(s.q)
            s.kv.AppendRopeDev(0, c["pos0"], q, s.K, s.V, THETA)
        else:
            s.kv.AppendRangeDev(0, c["pos0"], s.K, s.V, src_dtype=c["dtype"])
        s.kv.AttentionChunkDev(0, c["pos0"], q, s.out, s.scale, q_dtype=c["q_dtype"])
        return {"out": s.out, "q": q} if c["rope"] else {"out": s.out}
    if s.kind == "mla":
        s.m.AbsorbedAttentionDev(0, s.pos, s.qt, s.qrp, s.out, s.scale)
        return s.out
    if s.kind == "mla_layer":
        s.m.AttendAbsorbedDev(0, s.pos, s.q, s.w, CODE[s.c["wfmt"]], s.c["nope"], s.c["vdim"], s.out)
        return s.out
    for i, grp in enumerate(GROUPS):
        qr.matvec_group_dev([s.w[j] for j in grp], s.code, [s.mats[j][0] for j in grp], s.mats[grp[0]][1], s.x[i],
                            [s.out[j] for j in grp])
    return s.out


# ------------------------------------------------------------------ what a pass needs
def _wbytes(fmt, rows, cols):
    bs, bb = BLOCK[fmt]
    return rows * cols // bs * bb


def work(case):
    """K/V, queries, weights and outputs once each; 4 D flops per (query, key, head), 2 per weight."""
    c, k = case, case["kind"]
    if k == "decode":
        n, kvd, hd = sum(lengths(c)), c["kv"] * c["D"], c["heads"] * c["D"]
        return {"bytes": 2 * n * kvd * SIZE[c["dtype"]] + 8 * c["B"] * hd, "flops": 4 * n * hd}
    if k == "step":
        kvd, hd, dim, n = c["kv"] * c["D"], c["heads"] * c["D"], _step_dim(c), c["pos"] + 1
        mats = ((hd, dim), (kvd, dim), (kvd, dim), (dim, hd))
        b = sum(_wbytes(c["wfmt"], r, m) for r, m in mats) + 2 * n * kvd * SIZE[c["dtype"]] + 8 * dim
        f = sum(2 * r * m for r, m in mats) + 4 * n * hd
        return {"bytes": c["layers"] * b, "flops": c["layers"] * f}
    if k == "chunk":
        kvd, hd, nq = c["kv"] * c["D"], c["heads"] * c["D"], c["nq"]
        src = 4 if c["rope"] else SIZE[c["dtype"]]
        b = 2 * (c["pos0"] + nq) * kvd * SIZE[c["dtype"]] + 2 * nq * kvd * src + nq * hd * (SIZE[c["q_dtype"]] + 4)
        keys = nq * c["pos0"] + nq * (nq + 1) // 2
        return {"bytes": b + (8 * nq * hd if c["rope"] else 0), "flops": 4 * keys * hd}
    if k in ("mla", "mla_layer"):
        width = c["lora"] + c["rope_dim"]
        b, f = c["n"] * width * SIZE[c["dtype"]], 2 * c["heads"] * c["n"] * (width + c["lora"])
        if k == "mla":
            return {"bytes": b + 4 * c["heads"] * (width + c["lora"]), "flops": f}
        rows = c["heads"] * (c["nope"] + c["vdim"])
        return {"bytes": b + _wbytes(c["wfmt"], rows, c["lora"]) + 4 * c["heads"] * (c["nope"] + c["rope_dim"] + c["vdim"]),
                "flops": f + 2 * rows * c["lora"]}
    mats = _mats(c)
    b = sum(_wbytes(c["wfmt"], r, m) + 4 * c["nq"] * r for r, m in mats) + sum(4 * c["nq"] * mats[g[0]][1] for g in GROUPS)
    return {"bytes": b, "flops": 2 * c["nq"] * sum(r * m for r, m in mats)}


def tolerance(case):
    """MatVecs are specified to the bit (each format's own order of fp32 operations).  Attention is
    bounded by the cache type, about four times the distance from exact() that was measured: fp32
    sums 3e-7 to 1.3e-6; probabilities and split partials in 16 bits up to 2e-4 (f16) and 1.6e-3
    (bf16)."""
    if case["kind"] == "matvec":
        return "exact"
    return {"rel": {"f32": 5e-6, "f16": 1e-3, "bf16": 6e-3}[case["dtype"]]}


# ------------------------------------------------------------------ 64-bit results
def _attend(q, K, V, heads, kv, D, pos0, scale):
    """Causal attention of q [nq, heads * D] (query i sees keys 0..pos0 + i) over K, V [n, kv * D]."""
    nq, n = q.shape[0], K.shape[0]
    out = torch.empty(nq, heads * D, dtype=torch.float64, device="cuda")
    limit = torch.arange(pos0, pos0 + nq, device="cuda")[:, None]
    masked = torch.arange(n, device="cuda")[None, :] > limit if nq > 1 else None
    for h in range(heads):
        j = h * kv // heads
        s = q[:, h * D:(h + 1) * D] @ K[:, j * D:(j + 1) * D].double().t().contiguous() * scale
        if masked is not None:
            s.masked_fill_(masked, -math.inf)
        out[:, h * D:(h + 1) * D] = torch.softmax(s, -1) @ V[:, j * D:(j + 1) * D].double()
    return out


def _rope(x, D, pos0):
    """Rotate-half RoPE of rows at pos0.., with the fp32 angles that define it (position times fp32 frequency)."""
    n, half = x.shape[0], D // 2
    freq = torch.tensor([THETA ** (-2.0 * i / D) for i in range(half)], dtype=torch.float64).float()
    ang = (torch.arange(pos0, pos0 + n).float()[:, None] * freq[None, :]).double().cuda()[:, None, :]
    v = x.double().view(n, -1, D)
    a, b = v[..., :half], v[..., half:]
    return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], -1).view(n, -1)


def exact(case, seed):
    c, d, k = case, _inputs(case, seed), case["kind"]
    if k == "decode":
        out, at, scale = [], 0, 1.0 / math.sqrt(c["D"])
        for i, n in enumerate(lengths(c)):
            out.append(_attend(d["q"][i:i + 1].double(), d["K"][at:at + n], d["V"][at:at + n], c["heads"], c["kv"], c["D"],
                               n - 1, scale))
            at += n
        return torch.cat(out)
    if k == "step":
        kvd, hd, dim = c["kv"] * c["D"], c["heads"] * c["D"], _step_dim(c)
        out = []
        for l in range(c["layers"]):
            x, w = d["x"][l].double(), d["w"][l]
            q, kr, vr = (_decode(c["wfmt"], w[i], r, dim) @ x for i, r in ((0, hd), (1, kvd), (2, kvd)))
            t = TORCH[c["dtype"]]
            K = torch.cat([d["K"][l], _rope(kr[None], c["D"], c["pos"]).to(t)])
            V = torch.cat([d["V"][l], vr[None].to(t)])
            a = _attend(_rope(q[None], c["D"], c["pos"]), K, V, c["heads"], c["kv"], c["D"], c["pos"], 1.0 / math.sqrt(c["D"]))
            out.append(_decode(c["wfmt"], w[3], dim, hd) @ a[0])
        return out
    if k == "chunk":
        t, q, K = TORCH[c["dtype"]], d["q"], d["K"]
        if c["rope"]:
            q, K = _rope(q, c["D"], c["pos0"]), _rope(K, c["D"], c["pos0"])
        K, V = torch.cat([d["K0"], K.to(t)]), torch.cat([d["V0"], d["V"].to(t)])
        out = _attend(q.double(), K, V, c["heads"], c["kv"], c["D"], c["pos0"], 1.0 / math.sqrt(c["D"]))
        return {"out": out, "q": q} if c["rope"] else {"out": out}
    if k in ("mla", "mla_layer"):
        rows, L = d["rows"].double(), c["lora"]
        if k == "mla":
            qt, qrp, scale = d["qt"].double(), d["qrp"].double(), 1.0 / math.sqrt(192.0)
        else:
            H, nope, vdim = c["heads"], c["nope"], c["vdim"]
            w, q = _decode(c["wfmt"], d["w"], H * (nope + vdim), L).view(H, nope + vdim, L), d["q"].double()
            qt, qrp = torch.stack([q[h, :nope] @ w[h, :nope] for h in range(H)]), q[:, nope:]
            scale = 1.0 / math.sqrt(nope + c["rope_dim"])
        s = (qt @ rows[:, :L].t().contiguous() + qrp @ rows[:, L:].t().contiguous()) * scale
        u = torch.softmax(s, -1) @ rows[:, :L].contiguous()
        return u if k == "mla" else torch.stack([w[h, nope:] @ u[h] for h in range(H)])
    out = []
    for i, grp in enumerate(GROUPS):
        for j in grp:
            r, m = _mats(c)[j]
            out.append(d["x"][i].double() @ _decode(c["wfmt"], d["w"][j], r, m).t().contiguous())
    return out
