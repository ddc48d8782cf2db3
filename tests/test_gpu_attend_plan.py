"""Gathered attention at query counts on either side of the two-role kernel's first, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,n,heads,k", [(1, 128, 64, 70), (1, 129, 64, 70), (3, 43, 64, 1), (1, 255, 64, 640),
                                         (2, 33, 128, 161), (1, 129, 64, 2304), (1, 129, 64, 2305), (1, 130, 48, 90)])
def test_query_counts(gpu, b, n, heads, k):
    from dsv41.sparse_attention import sparse_attn
    g = torch.Generator(device="cuda").manual_seed(n + k)
    q = torch.randn(b, n, heads, 512, generator=g, device="cuda").bfloat16()
    kv = torch.randn(b, 700, 512, generator=g, device="cuda").bfloat16()
    idx = torch.randint(-40, 700, (b, n, k), generator=g, device="cuda", dtype=torch.int32).clamp(min=-1)
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


def _packed_decode(b, k, start, seed=5):
    """One token per sequence over the packed caches, as a function of a range of sequences; its ring too."""
    from dsv41 import _abi
    from dsv41.layers import precompute_freqs_cis
    g = torch.Generator(device="cuda").manual_seed(seed)
    ints = lambda lo, hi, *s: torch.randint(lo, hi, s, generator=g, device="cuda", dtype=torch.int32)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    wp, nb = min(start, 128), 900
    q, chunk, sink = rnd(b, 1, 64, 512).bfloat16(), rnd(b, 1, 512).bfloat16(), rnd(64)
    ring = torch.cat([rnd(b, 128, 512).to(torch.float8_e4m3fn).view(torch.uint8),
                      ints(126, 129, b, 128, 16).to(torch.uint8)], -1).contiguous()
    comp = torch.cat([ints(0, 256, b, nb, 256).to(torch.uint8), ints(40, 52, b, nb, 32).to(torch.uint8)], -1).contiguous()
    idx = (ints(0, nb, b, 1, k) + wp + 1).contiguous() if k else None
    cos, sin = precompute_freqs_cis(64, start + 1, 65536, 160000.0, 16.0, 32, 1)

    def run(lo, hi):
        r = ring[lo:hi].clone()
        o = _abi.sparse_mla_packed(q[lo:hi].contiguous(), r, chunk[lo:hi].contiguous(), comp[lo:hi].contiguous(), nb, sink,
                                   idx[lo:hi].contiguous() if k else None, 512 ** -0.5, 128, start, cos, sin, 64,
                                   write_ring=True, q_rd=64)
        return o, r
    return run


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
    run = _packed_decode(b, k, start)
    got, ring = run(0, b)
    for lo in (0, b - 128):
        o, r = run(lo, lo + 128)
        assert torch.equal(got[lo:lo + 128], o) and torch.equal(ring[lo:lo + 128], r)
