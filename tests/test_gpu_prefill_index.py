"""The chunk (8 or more queries) forms of the indexer against the one-query kernels: the same scores, bit for bit."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(b, n, heads, nb, seed, spare=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q = torch.randn(b, n, heads, 128, generator=g, device="cuda").bfloat16()
    w = torch.randn(b, n, heads, generator=g, device="cuda").bfloat16()
    k = torch.randn(b, nb + spare, 128, generator=g, device="cuda").bfloat16()
    return g, q, w, k


def _per_query(q, w, keys, start, ratio, cand):
    """Scores of each query by a call of its own (the one-query kernel, a workgroup per query)."""
    from dsv41 import _abi
    rows = []
    for s in range(q.shape[1]):
        c = None if cand is None else cand[:, s:s + 1].contiguous()
        rows.append(_abi.indexer_score(q[:, s:s + 1].contiguous(), w[:, s:s + 1].contiguous(), 0.07, keys, start + s,
                                       ratio, c))
    return torch.cat(rows, 1)


@pytest.mark.parametrize("b,n,heads,nb,start,ratio,keep", [
    (1, 8, 32, 1, 0, 1, 0.5),            # one key; most queries see it only
    (2, 9, 64, 63, 40, 1, 0.5),          # partial query group, partial chunk, causal edge inside the range
    (1, 15, 16, 64, 60, 1, 0.0),         # nothing kept
    (1, 17, 32, 2047, 8171, 4, 0.05),    # most 16-row tiles empty; odd nb: byte loads of the mask
    (2, 8, 64, 2048, 8184, 4, 0.5),      # one whole range, vector loads of the mask
    (1, 24, 32, 2064, 2040, 1, 1.0),     # everything kept; the last range holds 16 rows
    (1, 16, 32, 4101, 16400, 4, 0.3),    # several ranges, queries before and after the last key
])
def test_masked_chunk_scores_equal_per_query(gpu, b, n, heads, nb, start, ratio, keep):
    from dsv41 import _abi
    g, q, w, k = _inputs(b, n, heads, nb, nb + n, spare=3)
    keys = k[:, :nb]                     # a view of a longer cache
    cand = torch.rand(b, n, (nb + 7) // 8, generator=g, device="cuda").lt(keep).repeat_interleave(8, -1)[..., :nb]
    cand = cand.to(torch.uint8).mul_(255).contiguous()       # any non-zero byte keeps an entry
    got = _abi.indexer_score(q, w, 0.07, keys, start, ratio, cand)
    assert torch.equal(got, _per_query(q, w, keys, start, ratio, cand))
    assert torch.equal(_abi.indexer_score(q, w, 0.07, keys, start, ratio), _per_query(q, w, keys, start, ratio, None))


def test_masked_chunk_unaligned_mask(gpu):
    """A mask whose rows are whole 16-byte pieces but whose base is not aligned takes the byte loads."""
    from dsv41 import _abi
    g, q, w, k = _inputs(1, 10, 32, 256, 5)
    room = torch.zeros(10 * 256 + 3, dtype=torch.uint8, device="cuda")
    cand = room[3:].view(1, 10, 256)
    cand.copy_(torch.rand(1, 10, 256, generator=g, device="cuda").lt(0.2))
    got = _abi.indexer_score(q, w, 0.07, k, 300, 1, cand)
    assert torch.equal(got, _abi.indexer_score(q, w, 0.07, k, 300, 1, cand.clone()))


@pytest.mark.parametrize("n,nb", [(8, 16385), (64, 8192)])
def test_masked_selection_same_in_both_forms(gpu, n, nb):
    """Score + select, the form chunks take, against the fused form where that one serves the shape."""
    from dsv41 import _abi
    g, q, w, k = _inputs(1, n, 32, nb, 11)
    cand = torch.rand(1, n, (nb + 7) // 8, generator=g, device="cuda").lt(0.4).repeat_interleave(8, -1)[..., :nb]
    cand = cand.contiguous()
    two = _abi.topk_select(_abi.indexer_score(q, w, 0.07, k, nb - n, 1, cand), 128, nb - n, 1, 7)
    fused = _abi.indexer_topk(q, w, 0.07, k, nb - n, 1, 128, 7, cand)
    assert fused is not None and torch.equal(two, fused)


@pytest.mark.parametrize("b,n,heads,nb,start,ratio,keep", [
    (1, 8, 32, 1, 0, 1, None),           # one key; a query before it
    (2, 9, 64, 63, 40, 1, 0.5),          # partial query group, partial key block, causal edge inside it
    (1, 17, 16, 513, 700, 1, None),      # the range's waves get uneven shares
    (3, 11, 32, 2049, 2040, 1, 0.3),     # a last range of one key
    (1, 64, 32, 4101, 16388, 4, None),   # several ranges, queries before and after the last key
    (2, 13, 64, 1024, 4084, 4, 0.05),
])
def test_mxfp4_chunk_scores_equal_per_query(gpu, b, n, heads, nb, start, ratio, keep):
    from dsv41 import _abi
    g = torch.Generator(device="cuda").manual_seed(nb + n)

    def ints(lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)

    qc, qs = ints(0, 256, b, n, heads, 64), ints(118, 132, b, n, heads, 4)
    kc, ks = ints(0, 256, b, nb + 5, 64), ints(118, 132, b, nb + 5, 4)      # a longer cache
    w = torch.randn(b, n, heads, generator=g, device="cuda").bfloat16()
    cand = None
    if keep is not None:
        cand = torch.rand(b, n, nb, generator=g, device="cuda").lt(keep).to(torch.uint8).mul_(7).contiguous()
    got = _abi.indexer_score_mxfp4((qc, qs), w, 0.07, kc, ks, nb, start, ratio, cand)
    rows = []
    for s in range(n):                   # each query by a call of its own: the one-query kernel
        c = None if cand is None else cand[:, s:s + 1].contiguous()
        rows.append(_abi.indexer_score_mxfp4((qc[:, s:s + 1].contiguous(), qs[:, s:s + 1].contiguous()),
                                             w[:, s:s + 1].contiguous(), 0.07, kc, ks, nb, start + s, ratio, c))
    assert torch.equal(got, torch.cat(rows, 1))


@pytest.mark.parametrize("b,n,heads,nb,start,ratio,rb,keep", [
    (1, 8, 32, 1, 0, 1, 32, None),       # one key; a query before it
    (2, 9, 64, 63, 40, 1, 1, 0.5),       # partial query group, partial key chunk, causal edge inside it
    (1, 17, 16, 513, 700, 1, 32, 0.02),  # most 16-row tiles empty
    (3, 11, 32, 2049, 2040, 1, 1, 0.3),  # a last range of one key
    (1, 64, 32, 4101, 16388, 4, 32, None),
    (2, 13, 64, 1024, 4084, 4, 32, None),
])
def test_fp8_chunk_scores_equal_per_query(gpu, b, n, heads, nb, start, ratio, rb, keep):
    from dsv41 import _abi
    g, q, w, k = _inputs(b, n, heads, nb, nb + n, spare=5)
    codes = k.to(torch.float8_e4m3fn).view(torch.uint8)
    scales = torch.randint(118, 132, (b, (nb + 5 + rb - 1) // rb, 4), generator=g, device="cuda", dtype=torch.int32)
    scales = scales.to(torch.uint8)
    cand = None
    if keep is not None:
        cand = torch.rand(b, n, nb, generator=g, device="cuda").lt(keep).to(torch.uint8).contiguous()
    got = _abi.indexer_score_fp8(q, w, 0.07, codes, scales, rb, nb, start, ratio, cand)
    rows = []
    for s in range(n):                   # each query by a call of its own: the one-query kernel
        c = None if cand is None else cand[:, s:s + 1].contiguous()
        rows.append(_abi.indexer_score_fp8(q[:, s:s + 1].contiguous(), w[:, s:s + 1].contiguous(), 0.07, codes, scales,
                                           rb, nb, start + s, ratio, c))
    assert torch.equal(got, torch.cat(rows, 1))


# (queries, keys, start, ratio). Ranges: of 10 chunks in one piece; of 9 and 9; of 300 keys with one query per
# wave at 32 heads; of many even pieces with a short last one; masks read by vectors (1,104, 3,008) and by bytes.
RANGES = [(1700, 600, 0, 1), (1501, 1100, 350, 1), (1999, 300, 0, 1), (301, 3008, 2858, 1), (430, 1104, 889, 1),
          (77, 16500, 16462, 1)]
# Edges, over enough scores for the chunk kernels: one key, which the first query does not see at ratio 2;
# partial last query groups; a partial chunk with the causal edge inside; queries before and after the last key.
EDGES = [(3000, 1, 0, 2), (2001, 63, 40, 1), (1999, 64, 60, 1), (999, 2047, 7500, 4), (601, 4101, 16100, 4)]


@pytest.mark.parametrize("n,nb,start,ratio,keep", [(*c, keep) for keep in (None, 0.3) for c in RANGES + EDGES] +
                         [(*c, 0.0) for c in EDGES[:3]])
@pytest.mark.parametrize("heads", [16, 32, 64])
@pytest.mark.parametrize("fmt", ["bf16", "fp8", "mxfp4"])
def test_chunk_scores_equal_few_queries(gpu, fmt, keep, heads, n, nb, start, ratio):
    from dsv41 import _abi
    g, q, w, k = _inputs(1, n, heads, nb, nb + n)
    ints = lambda lo, hi, *s: torch.randint(lo, hi, s, generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)
    codes = k.to(torch.float8_e4m3fn).view(torch.uint8)
    scales = ints(118, 132, 1, (nb + 31) // 32, 4)
    q4, qs, k4, ks = ints(0, 256, 1, n, heads, 64), ints(118, 132, 1, n, heads, 4), ints(0, 256, 1, nb, 64), ints(118, 132, 1, nb, 4)
    cand = None if keep is None else torch.rand(1, n, nb, generator=g, device="cuda").lt(keep).contiguous()

    def run(lo, hi):
        part = lambda t: t[:, lo:hi].contiguous()
        c, ws = None if cand is None else part(cand), (part(w), 0.07)
        if fmt == "mxfp4":
            return _abi.indexer_score_mxfp4((part(q4), part(qs)), *ws, k4, ks, nb, start + lo, ratio, c)
        if fmt == "fp8":
            return _abi.indexer_score_fp8(part(q), *ws, codes, scales, 32, nb, start + lo, ratio, c)
        return _abi.indexer_score(part(q), *ws, k, start + lo, ratio, c)

    few = torch.cat([run(lo, min(lo + 7, n)) for lo in range(0, n, 7)], 1)
    assert torch.equal(run(0, n), few)
