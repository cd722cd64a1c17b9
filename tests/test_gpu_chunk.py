"""GPU parity of causal multi-query attention (chunked prefill, speculative verify).

Reference semantics: query i at position pos0+i equals a PagedKvCache.Attention
call at that position over rows 0..pos0+i (StreamingEngine.cs:831-836,
SpeculativeRunner.cs:85-93); the oracle is run on the exactly decoded 16-bit values.
16-bit caches run on MFMA tiles in the cache's own type (queries of another type as
hi + lo parts, P rounded to the cache type): tolerance max-abs <= 1e-3 and rel-L2
<= 5e-3 for bf16 caches, <= 1e-3 for fp16 caches.  Both sides' errors against fp64
are printed.
"""
import math

import numpy as np
import pytest

import qauntrunner_amd as qr
from oracle import oracle
from tests.util import assert_close, errors, to_dtype_bits

pytestmark = pytest.mark.gpu

TOL_REL = {"bf16": 5e-3, "f16": 1e-3}


def make(seed, n, kv_dim, dtype):
    rng = np.random.default_rng(seed)
    K = rng.standard_normal((n, kv_dim), dtype=np.float32)
    V = rng.standard_normal((n, kv_dim), dtype=np.float32)
    Kb, Kd = to_dtype_bits(K, dtype)
    Vb, Vd = to_dtype_bits(V, dtype)
    return Kb, Kd, Vb, Vd


def check_query(out_i, Kd, Vd, q_i, heads, kv_heads, D, scale, tol_rel, what):
    want = oracle.kv_attention(Kd, Vd, q_i, heads, kv_heads, D, scale)
    a, r = assert_close(out_i, want, 1e-3, tol_rel, what)
    f64 = oracle.kv_attention_f64(Kd, Vd, q_i, heads, kv_heads, D, scale)
    print(f"{what}: vs oracle max-abs {a:.2e} rel {r:.2e} | vs fp64 gpu {errors(out_i, f64)[1]:.2e} "
          f"oracle {errors(want, f64)[1]:.2e}")


def test_c3_chunked_prefill_bf16(gpu):
    """32 q heads / 8 kv heads / head_dim 128: 2048 bf16 queries after 6144 cached tokens."""
    heads, kv_heads, D, pos0, nq = 32, 8, 128, 6144, 2048
    n = pos0 + nq
    Kb, Kd, Vb, Vd = make(600, n, kv_heads * D, "bf16")
    qb, qd = to_dtype_bits(np.random.default_rng(601).standard_normal((nq, heads * D), dtype=np.float32), "bf16")
    scale = 1 / math.sqrt(D)
    with qr.PagedKvCache(1, heads, kv_heads, D, n, kv_dtype="bf16") as kv:
        kv.AppendRange(0, 0, Kb, Vb, src_dtype="bf16")
        out = kv.AttentionChunk(0, pos0, qb, scale, q_dtype="bf16")
    for i in (0, 1, 31, 63, 64, 255, 1000, 1337, 2047):
        check_query(out[i], Kd[:pos0 + i + 1], Vd[:pos0 + i + 1], qd[i], heads, kv_heads, D, scale,
                    TOL_REL["bf16"], f"C3 query {i}")
    # every query: causal attention recomputed in fp32 on the CPU (batched per kv head; a
    # plain fp32 formulation agrees with the oracle's op order to ~1e-6, far inside the
    # tolerance), at the same tolerances, query by query
    check_all_queries(out, Kd, Vd, qd, heads, kv_heads, D, pos0, scale, TOL_REL["bf16"], "C3")


def check_all_queries(out, Kd, Vd, qd, heads, kv_heads, D, pos0, scale, tol_rel, what):
    import torch

    nq, n = qd.shape[0], Kd.shape[0]
    G = heads // kv_heads
    K = torch.from_numpy(Kd).view(n, kv_heads, D)
    V = torch.from_numpy(Vd).view(n, kv_heads, D)
    Q = torch.from_numpy(qd).view(nq, heads, D)
    got = torch.from_numpy(np.ascontiguousarray(out)).view(nq, heads, D)
    seen = torch.arange(n)[None, :] > (pos0 + torch.arange(nq))[:, None]  # [nq, n]: past the query's position
    worst_abs, worst_rel = 0.0, 0.0
    for kvh in range(kv_heads):
        q = Q[:, kvh * G:(kvh + 1) * G, :]                        # [nq, G, D]
        s = torch.matmul(q, K[:, kvh, :].T.contiguous()) * scale  # [nq, G, n]
        s.masked_fill_(seen[:, None, :], float("-inf"))
        want = torch.matmul(torch.softmax(s, dim=-1), V[:, kvh, :].contiguous())  # [nq, G, D]
        g = got[:, kvh * G:(kvh + 1) * G, :]
        d = (g - want).reshape(nq, -1)
        abs_err = d.abs().max(dim=1).values
        rel_err = d.norm(dim=1) / want.reshape(nq, -1).norm(dim=1)
        worst_abs, worst_rel = max(worst_abs, float(abs_err.max())), max(worst_rel, float(rel_err.max()))
        bad = torch.nonzero((abs_err > 1e-3) | (rel_err > tol_rel)).flatten()
        assert bad.numel() == 0, f"{what}: kv head {kvh}, query {int(bad[0])}: max-abs {float(abs_err[bad[0]]):.2e} rel {float(rel_err[bad[0]]):.2e}"
    print(f"{what}, all {nq} queries vs fp32 CPU attention: worst max-abs {worst_abs:.2e}, worst rel-L2 {worst_rel:.2e}")


def test_c4_speculative_verify_fp16(gpu):
    """64 q heads / 8 kv heads: 8 draft queries at 131072..131079 over fp16 KV, causal among drafts."""
    heads, kv_heads, D, pos0, nq = 64, 8, 128, 131072, 8
    n = pos0 + nq
    Kb, Kd, Vb, Vd = make(700, n, kv_heads * D, "f16")
    qb, qd = to_dtype_bits(np.random.default_rng(701).standard_normal((nq, heads * D), dtype=np.float32), "f16")
    scale = 1 / math.sqrt(D)
    with qr.PagedKvCache(1, heads, kv_heads, D, n, kv_dtype="f16") as kv:
        kv.AppendRange(0, 0, Kb, Vb, src_dtype="f16")
        out = kv.AttentionChunk(0, pos0, qb, scale, q_dtype="f16")
        single = kv.Attention(0, pos0 + 3, qd[3], scale)
    for i in range(nq):
        check_query(out[i], Kd[:pos0 + i + 1], Vd[:pos0 + i + 1], qd[i], heads, kv_heads, D, scale,
                    TOL_REL["f16"], f"C4 verify draft {i}")
    assert_close(out[3], single, 1e-3, 1e-3, "verify draft 3 vs single decode call")


@pytest.mark.parametrize("dtype,heads,kv_heads,D,pos0,nq,q_dtype", [
    ("f16", 8, 8, 64, 0, 300, "f16"),        # prefill from scratch, group 1
    ("bf16", 16, 8, 128, 1000, 77, "bf16"),  # group 2, ragged query block
    ("f16", 64, 8, 128, 513, 40, "f32"),     # group 8, fp32 queries as hi + lo fp16
    ("bf16", 32, 4, 64, 255, 129, "bf16"),   # head_dim 64, crosses page boundaries
    ("f16", 4, 4, 128, 7, 1, "f16"),         # single query
    ("bf16", 32, 8, 128, 4000, 300, "f32"),  # fp32 queries as hi + lo bf16, two N tiles
    ("bf16", 8, 2, 64, 130, 1000, "f16"),    # fp16 queries into a bf16 cache, four N tiles
    ("f16", 16, 2, 128, 70000, 5, "f16"),    # few queries over a long cache: split-K, 3 stages
    # verify-sized blocks (one N tile: two waves per row group, one per 32-position half)
    ("f16", 64, 8, 64, 20, 8, "f32"),        # one tile of 28 positions: the second half all masked
                                             # (fp16: over 21 keys bf16's 8-bit P alone errs ~1.6e-3)
    ("f16", 32, 8, 128, 40, 8, "f16"),       # one tile of 48: the drafts' causal edge in the second half
    ("bf16", 64, 8, 128, 100, 8, "bf16"),    # two tiles, the last one partial
    ("bf16", 64, 8, 128, 5000, 8, "f32"),    # fp32 drafts as hi + lo bf16 over split keys
])
def test_chunk_mfma_shapes(gpu, dtype, heads, kv_heads, D, pos0, nq, q_dtype):
    n = pos0 + nq
    Kb, Kd, Vb, Vd = make(n + heads, n, kv_heads * D, dtype)
    qb, qd = to_dtype_bits(np.random.default_rng(n).standard_normal((nq, heads * D), dtype=np.float32), q_dtype)
    scale = 1 / math.sqrt(D)
    with qr.PagedKvCache(1, heads, kv_heads, D, n + 10, kv_dtype=dtype) as kv:
        kv.AppendRange(0, 0, Kb, Vb, src_dtype=dtype)
        out = kv.AttentionChunk(0, pos0, qb, scale, q_dtype=q_dtype)
    for i in sorted({0, nq // 2, nq - 1}):
        check_query(out[i], Kd[:pos0 + i + 1], Vd[:pos0 + i + 1], qd[i], heads, kv_heads, D, scale,
                    TOL_REL[dtype], f"{dtype} H{heads}/Hkv{kv_heads}/D{D} pos0 {pos0} query {i}")


def causal_f64(K, V, q, heads, kv_heads, D, pos0, scale):
    """All queries of a chunk in float64."""
    K, V, q = (np.asarray(x, np.float64) for x in (K, V, q))
    out = np.empty((q.shape[0], heads * D))
    seen = np.arange(K.shape[0])[None, :] <= pos0 + np.arange(q.shape[0])[:, None]
    for h in range(heads):
        j = slice(h * kv_heads // heads * D, (h * kv_heads // heads + 1) * D)
        s = np.where(seen, q[:, h * D:(h + 1) * D] @ K[:, j].T * scale, -np.inf)
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h * D:(h + 1) * D] = p @ V[:, j] / p.sum(1, keepdims=True)
    return out


@pytest.mark.parametrize("dtype,heads,kv_heads,D,pos0,nq,q_dtype", [
    ("f32", 32, 8, 96, 0, 2, "f32"),         # 8 rows per kv head: the fewest, one tile of 2 keys
    ("f32", 32, 8, 96, 33, 8, "f32"),        # 32 rows, two position halves, second tile of 9 keys
    ("f32", 32, 8, 64, 0, 65, "f32"),        # the fewest queries that need no key bytes
    ("f32", 32, 8, 128, 5000, 9, "f32"),     # 36 rows, keys split
    ("f32", 32, 8, 128, 0, 333, "f32"),      # from scratch: every tile masked for some block
    ("f32", 28, 4, 128, 255, 75, "bf16"),    # group 7, 16-bit queries, crosses a page
    ("f32", 24, 8, 96, 1000, 200, "f32"),    # group 3, head_dim 96 (8-byte V reads)
    ("f32", 16, 16, 256, 300, 67, "f16"),    # group 1, head_dim 256
    ("f32", 64, 1, 64, 7, 66, "f32"),        # 64 heads on one kv head
    ("f32", 32, 8, 64, 700, 600, "f32"),     # 64 rows a workgroup (no position halves), keys split
    ("f16", 24, 8, 96, 500, 130, "f16"),     # 16-bit pages, token-major
    ("bf16", 32, 8, 96, 90, 40, "f32"),
    ("bf16", 64, 8, 256, 250, 70, "bf16"),
    ("f16", 8, 2, 256, 9000, 7, "f32"),
    ("f32", 32, 8, 128, 3000, 5, "f32"),     # 20 rows over split keys, from the byte line up
    # groups above 32: always 64 rows a workgroup, one query each
    ("f32", 48, 1, 96, 0, 70, "f32"),        # unsplit
    ("f32", 40, 1, 128, 900, 70, "f32"),     # split
    ("f32", 64, 1, 128, 0, 100, "bf16"),
    ("f32", 64, 1, 256, 0, 66, "f32"),
    ("f32", 33, 1, 256, 2000, 70, "f32"),
    ("bf16", 64, 1, 96, 30, 40, "bf16"),
    ("f16", 40, 1, 256, 3000, 75, "f32"),
    ("f32", 24, 8, 256, 1000, 300, "f32"),   # 64 rows of 21 queries, split
    ("f32", 32, 8, 128, 700, 300, "f32"),
    ("f32", 16, 16, 256, 100, 140, "f16"),   # group 1, head_dim 256, past its line
    ("bf16", 16, 16, 256, 1000, 64, "f32"),
])
def test_chunk_f32_tiles(gpu, dtype, heads, kv_heads, D, pos0, nq, q_dtype):
    """fp32 arithmetic over the exactly decoded cache: fp32 sums over up to 5,000 keys, 5e-6
    relative (2^-24 times the square root of the terms, over the cancellation of the sum)."""
    n = pos0 + nq
    Kb, Kd, Vb, Vd = make(n + heads, n, kv_heads * D, dtype)
    qb, qd = to_dtype_bits(np.random.default_rng(n).standard_normal((nq, heads * D), dtype=np.float32), q_dtype)
    scale = 1 / math.sqrt(D)
    with qr.PagedKvCache(1, heads, kv_heads, D, n + 10, kv_dtype=dtype) as kv:
        kv.AppendRange(0, 0, Kb, Vb, src_dtype=dtype)
        out = kv.AttentionChunk(0, pos0, qb, scale, q_dtype=q_dtype)
    want = causal_f64(Kd, Vd, qd, heads, kv_heads, D, pos0, scale)
    for i in range(nq):
        a, r = errors(out[i], want[i])
        assert r <= 5e-6, f"query {i}: rel-L2 {r:.2e} max-abs {a:.2e}"


@pytest.mark.parametrize("dtype,heads,kv_heads,D,nq", [
    ("f32", 8, 2, 64, 70), ("f32", 8, 2, 128, 100), ("bf16", 8, 4, 96, 40), ("f16", 8, 8, 256, 300),
    # 64 rows a workgroup: unsplit, and split
    ("f32", 64, 1, 96, 70), ("f32", 40, 1, 128, 100), ("f32", 33, 1, 256, 75), ("f16", 64, 1, 96, 300),
    ("f32", 32, 8, 64, 600), ("bf16", 40, 1, 256, 290),
])
def test_chunk_f32_tiles_unseen_infinities(gpu, dtype, heads, kv_heads, D, nq):
    """An infinite V reaches the queries that see its position and no other."""
    Kb, Kd, Vb, Vd = make(3, nq, kv_heads * D, dtype)
    bad = nq - 2
    Vi, _ = to_dtype_bits(np.where(np.arange(nq)[:, None] == bad, np.float32(np.inf), Vd), dtype)
    q = np.random.default_rng(4).standard_normal((nq, heads * D), dtype=np.float32)
    out = {}
    for name, v in (("plain", Vb), ("inf", Vi)):
        with qr.PagedKvCache(1, heads, kv_heads, D, nq, kv_dtype=dtype) as kv:
            kv.AppendRange(0, 0, Kb, v, src_dtype=dtype)
            out[name] = kv.AttentionChunk(0, 0, q, 1 / math.sqrt(D))
    for i in range(bad):
        assert errors(out["inf"][i], out["plain"][i])[1] <= 5e-6, i
    assert np.all(out["inf"][bad:] == np.inf)


@pytest.mark.parametrize("dtype,heads,kv_heads,D,pos0,nq", [
    ("f32", 16, 4, 64, 0, 500),
    ("f32", 32, 8, 128, 0, 300),
    ("f32", 32, 8, 128, 1000, 200),
    ("f32", 16, 16, 256, 0, 300),
    ("bf16", 24, 8, 96, 0, 300),
    ("f16", 32, 8, 256, 0, 300),
])
def test_chunk_f32_tiles_error_of_decode_entries(gpu, dtype, heads, kv_heads, D, pos0, nq):
    """The distance from 64-bit results is no larger than that of one decode entry per query: 5%
    for the spread from seed to seed (1 to 3% over three seeds of these shapes)."""
    n = pos0 + nq
    Kb, Kd, Vb, Vd = make(n + heads, n, kv_heads * D, dtype)
    q = np.random.default_rng(n).standard_normal((nq, heads * D), dtype=np.float32) * np.float32(1.5)
    scale = 1 / math.sqrt(D)
    with qr.PagedKvCache(1, heads, kv_heads, D, n, kv_dtype=dtype) as kv:
        kv.AppendRange(0, 0, Kb, Vb, src_dtype=dtype)
        tiles = kv.AttentionChunk(0, pos0, q, scale)
        entries = np.concatenate([kv.AttentionBatch(0, [0] * len(r), list(r), q[r.start - pos0:r.stop - pos0], scale)
                                  for r in (range(p, min(p + 64, n)) for p in range(pos0, n, 64))])
    want = causal_f64(Kd, Vd, q, heads, kv_heads, D, pos0, scale)
    a, b = (np.linalg.norm(x.reshape(want.shape) - want) / np.linalg.norm(want) for x in (tiles, entries))
    print(f"tiles {a:.3e} entries {b:.3e}")
    assert a <= 1.05 * b


@pytest.mark.parametrize("dtype,heads,kv_heads,D", [("f32", 8, 2, 64), ("f32", 16, 16, 128), ("f32", 16, 8, 256),
                                                     ("bf16", 24, 8, 96)])
def test_chunk_f32_tiles_large_values(gpu, dtype, heads, kv_heads, D):
    """V near the top of the range.  Positions 0 to 31 have score 0, position 40 one of 7.5 log2
    units above and the others none to speak of, so a weight against any earlier maximum would
    overflow (2^7.5 x 5e36) where weights of at most 1 add up to 33 at most (1.7e38)."""
    nq, scale, v = 66, 1 / math.sqrt(D), 5e36
    K = np.full((nq, kv_heads * D), -100 / (D * scale), np.float32)
    K[:32] = 0
    K[40] = 7.5 * math.log(2) / (D * scale)
    Kb, _ = to_dtype_bits(K, dtype)
    Vb, Vd = to_dtype_bits(np.full((nq, kv_heads * D), v, np.float32), dtype)
    q = np.ones((nq, heads * D), np.float32)
    with qr.PagedKvCache(1, heads, kv_heads, D, nq, kv_dtype=dtype) as kv:
        kv.AppendRange(0, 0, Kb, Vb, src_dtype=dtype)
        out = kv.AttentionChunk(0, 0, q, scale)
    assert np.all(np.abs(out / Vd[0, 0] - 1) <= 5e-6)  # the fp32 sums' bound of the tests above


@pytest.mark.parametrize("dtype,heads,kv_heads,D,pos0,warm,nq", [
    ("f32", 32, 8, 128, 700, 1300, 300),    # the larger call is unsplit, the smaller wants three splits
    ("f16", 24, 8, 96, 1500, 1200, 70),
    ("f16", 24, 8, 128, 700, 1400, 300),    # 16-bit tiles of a group of three
])
def test_chunk_captured_after_a_larger_call(gpu, dtype, heads, kv_heads, D, pos0, warm, nq):
    """A captured chunk that wants more splits than any call before it had uses fewer, as the
    decode entries did not need a larger workspace either; every replay equals the eager result
    within the tolerance of the tiles."""
    import torch

    n = pos0 + warm
    Kb, _, Vb, _ = make(n, n, kv_heads * D, dtype)
    q = torch.from_numpy(np.random.default_rng(n).standard_normal((warm, heads * D), dtype=np.float32)).to(gpu)
    out, eager = torch.empty_like(q), torch.empty_like(q[:nq])
    scale = 1 / math.sqrt(D)
    with qr.PagedKvCache(1, heads, kv_heads, D, n, kv_dtype=dtype) as kv:
        kv.AppendRange(0, 0, Kb, Vb, src_dtype=dtype)
        kv.AttentionChunkDev(0, pos0, q, out, scale)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            kv.AttentionChunkDev(0, pos0, q[:nq], out[:nq], scale)
        results = []
        for _ in range(3):
            out.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            results.append(out[:nq].cpu().numpy())
        kv.AttentionChunkDev(0, pos0, q[:nq], eager, scale)
        torch.cuda.synchronize()
        del graph
    for r in results:
        assert errors(r, eager.cpu().numpy())[1] <= 2e-5


@pytest.mark.parametrize("dtype,heads,kv_heads,D,pos0,nq,q_dtype", [
    ("f16", 28, 4, 128, 0, 130, "f16"),      # group 7: 18 queries fill 126 of a block's 128 rows
    ("bf16", 24, 8, 64, 300, 131, "f32"),    # group 3, hi + lo queries
    ("bf16", 24, 8, 128, 5000, 9, "bf16"),   # few queries over few keys: decode entries
    ("bf16", 24, 8, 128, 7000, 9, "bf16"),   # one N tile, past the line of few queries
    ("f16", 20, 4, 64, 1000, 140, "f32"),    # group 5
    ("f16", 63, 1, 128, 5, 133, "f16"),      # group 63: one query per block of 64 rows, two of 128
])
def test_chunk_mfma_uneven_groups(gpu, dtype, heads, kv_heads, D, pos0, nq, q_dtype):
    """P (and fp32 queries) in hi + lo parts: about 22 (f16) and 16 (bf16) bits of each product's
    weight, 2e-5 and 2e-4 relative with the parts' own rounding (2^-16 times a few)."""
    n = pos0 + nq
    Kb, Kd, Vb, Vd = make(n + heads, n, kv_heads * D, dtype)
    qb, qd = to_dtype_bits(np.random.default_rng(n).standard_normal((nq, heads * D), dtype=np.float32), q_dtype)
    scale = 1 / math.sqrt(D)
    with qr.PagedKvCache(1, heads, kv_heads, D, n + 10, kv_dtype=dtype) as kv:
        kv.AppendRange(0, 0, Kb, Vb, src_dtype=dtype)
        out = kv.AttentionChunk(0, pos0, qb, scale, q_dtype=q_dtype)
    want = causal_f64(Kd, Vd, qd, heads, kv_heads, D, pos0, scale)
    for i in range(nq):
        a, r = errors(out[i], want[i])
        assert r <= {"f16": 2e-5, "bf16": 2e-4}[dtype], f"query {i}: rel-L2 {r:.2e} max-abs {a:.2e}"


@pytest.mark.parametrize("dtype,heads,kv_heads,D,pos0,nq,bad", [
    ("f16", 24, 8, 64, 0, 133, 70),       # the second of four query blocks, a split per tile
    ("f16", 28, 4, 128, 0, 140, 138),     # the last block: two queries see it
    ("bf16", 28, 4, 64, 500, 129, 510),   # the first block, splits of two tiles
    ("f16", 28, 4, 128, 0, 1200, 600),    # unsplit: masked and unmasked tiles in one workgroup
    ("bf16", 24, 8, 128, 300, 131, 372),
    ("f16", 24, 8, 128, 7000, 9, 7004),   # one N tile: two waves per row group, half a tile each
    ("bf16", 28, 4, 64, 13000, 18, 13001),
])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_chunk_mfma_uneven_groups_unseen_infinities(gpu, dtype, heads, kv_heads, D, pos0, nq, bad, value):
    """A V row that is not finite reaches the queries that see its position and no other: those
    give the same results as without it, within the tolerance of the uneven groups."""
    n = pos0 + nq
    Kb, Kd, Vb, Vd = make(n + heads, n, kv_heads * D, dtype)
    Vi, _ = to_dtype_bits(np.where(np.arange(n)[:, None] == bad, np.float32(value), Vd), dtype)
    q = np.random.default_rng(4).standard_normal((nq, heads * D), dtype=np.float32)
    out = {}
    for name, v in (("plain", Vb), ("bad", Vi)):
        with qr.PagedKvCache(1, heads, kv_heads, D, n, kv_dtype=dtype) as kv:
            kv.AppendRange(0, 0, Kb, v, src_dtype=dtype)
            out[name] = kv.AttentionChunk(0, pos0, q, 1 / math.sqrt(D))
    for i in range(bad - pos0):
        assert errors(out["bad"][i], out["plain"][i])[1] <= {"f16": 2e-5, "bf16": 2e-4}[dtype], f"query {i}"
    assert not np.isfinite(out["bad"][bad - pos0:]).any()


@pytest.mark.parametrize("scale", [0.0, -0.09])
@pytest.mark.parametrize("dtype,heads,kv_heads,D,pos0,nq,q_dtype", [
    ("f16", 28, 4, 128, 0, 140, "f16"),
    ("bf16", 24, 8, 64, 300, 131, "f32"),
    ("f16", 24, 8, 128, 7000, 9, "f32"),
    ("bf16", 32, 8, 128, 100, 70, "bf16"),
    ("f16", 64, 8, 64, 900, 6, "f32"),
])
def test_chunk_mfma_scale_zero_and_negative(gpu, dtype, heads, kv_heads, D, pos0, nq, q_dtype, scale):
    """Scale 0 is the mean of the rows seen so far, a negative one favours the opposite keys."""
    n = pos0 + nq
    Kb, Kd, Vb, Vd = make(n + heads, n, kv_heads * D, dtype)
    qb, qd = to_dtype_bits(np.random.default_rng(n).standard_normal((nq, heads * D), dtype=np.float32), q_dtype)
    with qr.PagedKvCache(1, heads, kv_heads, D, n, kv_dtype=dtype) as kv:
        kv.AppendRange(0, 0, Kb, Vb, src_dtype=dtype)
        out = kv.AttentionChunk(0, pos0, qb, scale, q_dtype=q_dtype)
    want = causal_f64(Kd, Vd, qd, heads, kv_heads, D, pos0, scale)
    for i in range(nq):
        assert errors(out[i], want[i])[1] <= TOL_REL[dtype], f"query {i}"


def test_chunk_mfma_uneven_groups_sum_small_weights(gpu):
    """Row sums of uneven groups are of the fp32 weights: position 0 has weight 1 and each of up
    to 4,143 others 2^-25.2, which fp16 hi + lo parts drop (below half of 2^-24) although they
    add up to 1.1e-4.  V cancels but at position 0, so the output is that row over the sum."""
    heads, kv_heads, D, pos0, nq = 24, 8, 64, 2800, 1344  # keys unsplit
    n = pos0 + nq
    K = np.zeros((n, kv_heads * D), np.float32)
    K[0] = np.float16(25.2 * math.log(2) / 8)  # score 8 K log2(e) log2 units above the others
    V = np.where(np.arange(n)[:, None] % 2 == 0, np.float32(1), np.float32(-1)) * np.ones((1, kv_heads * D), np.float32)
    Kb, Kd = to_dtype_bits(K, "f16")
    Vb, Vd = to_dtype_bits(V, "f16")
    q = np.ones((nq, heads * D), np.float32)
    with qr.PagedKvCache(1, heads, kv_heads, D, n, kv_dtype="f16") as kv:
        kv.AppendRange(0, 0, Kb, Vb, src_dtype="f16")
        out = kv.AttentionChunk(0, pos0, q, 1 / 8)
    want = causal_f64(Kd, Vd, q, heads, kv_heads, D, pos0, 1 / 8)
    for i in range(nq):
        assert errors(out[i], want[i])[1] <= 2e-5, f"query {i}"
