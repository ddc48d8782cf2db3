"""The index query prologue over a prompt's rows (wider pieces per thread) against the same tokens a few at a time."""

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
