"""Rope prologues over many rows (wider pieces per thread) against the same tokens a few at a time."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,n,heads,d,rd", [(1, 2048, 32, 128, 64), (2, 1025, 32, 128, 64), (1, 1030, 64, 128, 40),
                                            (1, 9000, 16, 64, 24)])
def test_prompt_rows_equal_few_tokens(gpu, b, n, heads, d, rd):
    """rd 64: the rope tail starts on a thread's piece; 40 and 24: inside one."""
    from dsv41 import _abi
    from dsv41.layers import precompute_freqs_cis
    g = torch.Generator(device="cuda").manual_seed(n)
    q = torch.randn(b, n, heads, d, generator=g, device="cuda").mul_(3).bfloat16()
    q[0, 1, 0] = 0.0
    q[0, 2, 0, ::5] = 5.0                # ties of the 4-bit grid at scale 1
    q[0, 3, 0, 7] = float("inf")
    cos, sin = precompute_freqs_cis(rd, n + 50, 65536, 160000.0, 16.0, 32, 1)
    few, codes, scales = [], [], []
    for s in range(0, n, 100):
        part = q[:, s:s + 100].clone()      # prepared in place
        if d == 128:
            c, x = _abi.index_q_prep_mxfp4(part, cos, sin, rd, 50 - 9 + s)
            codes.append(c)
            scales.append(x)
        _abi.index_q_prep(part, cos, sin, rd, 50 - 9 + s)
        few.append(part)
    if d == 128:
        c, x = _abi.index_q_prep_mxfp4(q, cos, sin, rd, 50 - 9)
        assert torch.equal(c, torch.cat(codes, 1)) and torch.equal(x, torch.cat(scales, 1))
    _abi.index_q_prep(q, cos, sin, rd, 50 - 9)
    assert torch.equal(q.view(torch.int16), torch.cat(few, 1).view(torch.int16))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,heads,d,rd,inverse", [(16400, 1, 512, 64, False), (260, 64, 512, 64, True), (33000, 1, 256, 40, True)])
def test_rope_tail_of_many_rows(gpu, dt, n, heads, d, rd, inverse):
    from dsv41 import _abi
    from dsv41.layers import precompute_freqs_cis
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(1, n, heads, d, generator=g, device="cuda").to(dt)
    cos, sin = precompute_freqs_cis(rd, n + 50, 65536, 160000.0, 16.0, 32, 1)
    few = [_abi.rope_tail(x[:, s:s + 4000 // heads].contiguous(), rd, cos, sin, 7 + s, 1, inverse)
           for s in range(0, n, 4000 // heads)]
    assert torch.equal(_abi.rope_tail(x, rd, cos, sin, 7, 1, inverse), torch.cat(few, 1))


@pytest.mark.parametrize("rb,g0,n,rd", [(1, 3, 16390, 64), (32, 0, 16400, 64), (32, 45, 16391, 64), (32, 64, 16385, 40)])
def test_fp8_cache_write_of_many_rows(gpu, rb, g0, n, rd):
    """rb 32: the row that opens a block sets its scale; g0 45 starts inside one, the pieces below too."""
    from dsv41 import _abi
    from dsv41.layers import precompute_freqs_cis
    g = torch.Generator(device="cuda").manual_seed(n)
    lat = torch.randn(1, n, 512, generator=g, device="cuda").mul_(2).bfloat16()
    cos, sin = precompute_freqs_cis(rd, 4 * (g0 + n), 65536, 160000.0, 16.0, 32, 1)
    rows = g0 + n + 5
    new = lambda: (torch.zeros(1, rows, 512, dtype=torch.uint8, device="cuda"),
                   torch.full((1, (rows + rb - 1) // rb, 16), 126, dtype=torch.uint8, device="cuda"))
    (codes, scales), (codes_few, scales_few) = new(), new()
    _abi.comp_write_fp8(lat, codes, scales, g0, 4, cos, sin, rd, rb)
    for s in range(0, n, 3001):
        _abi.comp_write_fp8(lat[:, s:s + 3001].contiguous(), codes_few, scales_few, g0 + s, 4, cos, sin, rd, rb)
    assert torch.equal(codes, codes_few) and torch.equal(scales, scales_few)
