"""Gathered attention at query counts on either side of the two-role kernel's first, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,n,heads,k", [(1, 128, 64, 70), (1, 129, 64, 70), (3, 43, 64, 1), (1, 255, 64, 640),
                                         (2, 33, 128, 161), (1, 129, 64, 2304), (1, 129, 64, 2305), (1, 130, 48, 90)])
def test_query_counts(gpu, b, n, heads, k):
    """Channels 500 and up are 0 in the queries and in all rows but one per list, which holds 200 there: with
    k rows of about equal weight that one is 200 / k of the output, so losing or repeating it, wherever it
    stands (steps' edges and the last entry among the places), is far outside the bound."""
    from dsv41.sparse_attention import sparse_attn
    g = torch.Generator(device="cuda").manual_seed(n + k)
    q = torch.randn(b, n, heads, 512, generator=g, device="cuda").bfloat16()
    kv = torch.randn(b, 700, 512, generator=g, device="cuda").bfloat16()
    q[..., 500:] = 0
    kv[..., 500:] = 0
    kv[:, 600:, 500:] = 200
    idx = torch.randint(-40, 600, (b, n, k), generator=g, device="cuda", dtype=torch.int32).clamp(min=-1)
    s = torch.arange(n, device="cuda")
    edges = torch.tensor([k - 1, 0, min(31, k - 1), min(32, k - 1), k // 2], device="cuda")
    place = torch.where(s % 2 == 0, edges[(s // 2) % 5], (s * 37) % k)
    idx.scatter_(2, place[None, :, None].expand(b, n, 1), (600 + s % 100).int()[None, :, None].expand(b, n, 1))
    sink = torch.randn(heads, generator=g, device="cuda")
    got = sparse_attn(q, kv, sink, idx, 512 ** -0.5).double()
    for i in range(b):
        for s in range(0, n, 32):
            ids = idx[i, s:s + 32].long()
            rows = kv[i].double()[ids.clamp(min=0)]
            logits = (q[i, s:s + 32].double() @ rows.transpose(1, 2)) * 512 ** -0.5
            logits = logits.masked_fill((ids < 0)[:, None], float("-inf"))
            full = torch.cat([logits, sink.double()[None, :, None].expand(ids.shape[0], -1, 1)], -1)
            p = torch.softmax(full, -1)[..., :-1]
            want, mass = p @ rows, p @ rows.abs()
            # weights and their sum from bf16 (2 x 2**-9), split partials and the output rounded to bf16 (2 x 2**-9)
            bound = 2 ** -7 * mass + 2 ** -8 * want.abs()
            assert bool(((got[i, s:s + 32] - want).abs() <= bound).all())
            assert bool((want[..., 500:] > 8 * bound[..., 500:]).all())      # the lone row would be missed


@pytest.mark.parametrize("most,fewer", [(200, (200, 128, 100)), (255, (129, 64))])
def test_workspace_of_the_most_queries_serves_fewer(gpu, most, fewer):
    from dsv41 import _abi
    from dsv41.sparse_attention import sparse_attn
    k = 640
    ws = torch.empty(_abi.mla_workspace_bytes(1, most, 64, 512, k, torch.bfloat16), dtype=torch.uint8, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(most)
    kv = torch.randn(1, 700, 512, generator=g, device="cuda").bfloat16()
    sink = torch.randn(64, generator=g, device="cuda")
    for n in fewer:
        q = torch.randn(1, n, 64, 512, generator=g, device="cuda").bfloat16()
        idx = torch.randint(0, 700, (1, n, k), generator=g, device="cuda", dtype=torch.int32)
        out = torch.empty_like(q)
        _abi._call("dsv41_sparse_attn", _abi._ptr(q), _abi._ptr(kv), _abi._ptr(sink), _abi._ptr(idx), _abi._ptr(out),
                   1, n, 64, 512, 700, k, 512 ** -0.5, _abi.dtype_code(q, "q"), _abi._ptr(ws), ws.numel(),
                   _abi._stream(q))
        assert torch.equal(out, sparse_attn(q, kv, sink, idx, 512 ** -0.5))


def _decode(fmt, b, k, start, seed=5):
    """One token per sequence over the caches of a format, as a function of a range of sequences; its ring too."""
    from dsv41 import _abi
    from dsv41.layers import precompute_freqs_cis
    g = torch.Generator(device="cuda").manual_seed(seed)
    ints = lambda lo, hi, *s: torch.randint(lo, hi, s, generator=g, device="cuda", dtype=torch.int32)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    wp, nb = min(start, 128), 900
    q, chunk, sink = rnd(b, 1, 64, 512).bfloat16(), rnd(b, 1, 512).bfloat16(), rnd(64)
    ring, comp = rnd(b, 128, 512).bfloat16(), rnd(b, nb, 512).bfloat16()
    scales = ints(126, 129, b, (nb + 31) // 32, 16).to(torch.uint8)
    if fmt == "fp8":
        comp = comp.to(torch.float8_e4m3fn).view(torch.uint8)
    elif fmt == "packed":
        ring = torch.cat([ring.to(torch.float8_e4m3fn).view(torch.uint8), ints(126, 129, b, 128, 16).to(torch.uint8)],
                         -1).contiguous()
        comp = torch.cat([ints(0, 256, b, nb, 256).to(torch.uint8), ints(40, 52, b, nb, 32).to(torch.uint8)], -1).contiguous()
    idx = None
    if k:                                # distinct entries: each one counts once
        idx = (torch.rand(b, 1, nb, generator=g, device="cuda").argsort(-1)[..., :k] + wp + 1).int().contiguous()
    cos, sin = precompute_freqs_cis(64, start + 1, 65536, 160000.0, 16.0, 32, 1)

    def run(lo, hi):
        part = lambda t: t[lo:hi].contiguous()
        r = part(ring).clone()
        tail = (nb, sink, part(idx) if k else None, 512 ** -0.5, 128, start, cos, sin, 64)
        kw = dict(write_ring=True, q_rd=64)
        if fmt == "packed":
            o = _abi.sparse_mla_packed(part(q), r, part(chunk), part(comp), *tail, **kw)
        elif fmt == "fp8":
            o = _abi.sparse_mla_fp8(part(q), r, part(chunk), part(comp), part(scales), 32, *tail, **kw)
        else:
            o = _abi.sparse_mla(part(q), r, part(chunk), part(comp), *tail, **kw)
        return o, r
    return run, chunk


@pytest.mark.parametrize("b", [129, 200])
@pytest.mark.parametrize("fmt", ["bf16", "fp8", "packed"])
def test_decode_forms_against_split_lists(gpu, fmt, b):
    """One token of 129 and of 200 sequences on the two-role kernel against 64 sequences at a time, whose lists
    are split: per sequence and head the two differ by bf16 roundings of the weights, the partials and the
    output (about 2**-8 of its norm together); one entry of 640 lost is 1 / sqrt(640), 4 %, of it."""
    run, chunk = _decode(fmt, b, 512, 8200)
    got, ring = run(0, b)
    few = [run(lo, min(lo + 64, b)) for lo in range(0, b, 64)]
    want = torch.cat([o for o, _ in few]).double()
    assert bool(((got.double() - want).norm(dim=-1) <= 2 ** -6 * want.norm(dim=-1)).all())
    assert torch.equal(ring, torch.cat([r for _, r in few]))
    if fmt != "packed":
        assert torch.equal(ring[:, 8200 % 128], chunk[:, 0])


@pytest.mark.parametrize("n,heads", [(129, 64), (255, 64), (65, 128)])
@pytest.mark.parametrize("k", [1, 32])
def test_lists_of_one_step_run_as_for_fewer_queries(gpu, n, heads, k):
    """No list to split and nothing to combine: the same kernel, bit for bit, as at 128 workgroups."""
    from dsv41.sparse_attention import sparse_attn
    g = torch.Generator(device="cuda").manual_seed(n + k)
    q = torch.randn(1, n, heads, 512, generator=g, device="cuda").bfloat16()
    kv = torch.randn(1, 300, 512, generator=g, device="cuda").bfloat16()
    idx = torch.randint(0, 300, (1, n, k), generator=g, device="cuda", dtype=torch.int32)
    sink = torch.randn(heads, generator=g, device="cuda")
    got = sparse_attn(q, kv, sink, idx, 512 ** -0.5)
    for part in torch.arange(n).split(8192 // heads):
        sub = slice(int(part[0]), int(part[-1]) + 1)
        assert torch.equal(got[:, sub], sparse_attn(q[:, sub].contiguous(), kv, sink, idx[:, sub].contiguous(), 512 ** -0.5))


@pytest.mark.parametrize("b,k,start", [(129, 0, 31), (129, 128, 8192), (150, 192, 8192), (192, 320, 8192)])
def test_packed_lists_run_as_for_128_sequences(gpu, b, k, start):
    run, _ = _decode("packed", b, k, start)
    got, ring = run(0, b)
    for lo in (0, b - 128):
        o, r = run(lo, lo + 128)
        assert torch.equal(got[lo:lo + 128], o) and torch.equal(ring[lo:lo + 128], r)
