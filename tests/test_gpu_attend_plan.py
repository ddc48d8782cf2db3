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
