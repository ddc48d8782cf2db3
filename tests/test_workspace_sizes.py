"""Workspace sizes are host arithmetic: one sized for the largest batch has to serve every smaller one."""

from __future__ import annotations

import pytest


@pytest.mark.parametrize("nb,k", [(16385, 512), (20000, 1024), (32768, 512), (32768, 2048), (32769, 512),
                                  (65536, 512), (65536, 3000), (131072, 1024), (400000, 64)])
def test_topk_workspace_never_falls_with_rows(nb, k):
    from dsv41 import _abi
    sizes = [_abi.topk_workspace_bytes(r, nb, k) for r in list(range(1, 700)) + [2048, 8192, 65536]]
    assert sizes == sorted(sizes)


def test_topk_rows_from_which_one_workgroup_selects_a_row():
    """The last row count that still takes two stages is the one whose workspace is the largest."""
    from dsv41 import _abi
    for nb, k, last in [(24576, 512, 63), (24577, 1024, 79), (32768, 64, 79), (32768, 1025, 63), (40000, 512, 127)]:
        sizes = [_abi.topk_workspace_bytes(r, nb, k) for r in range(1, 128)]
        assert sizes.index(max(sizes)) + 1 == last, (nb, k)


@pytest.mark.parametrize("heads,most", [(64, 255), (64, 200), (64, 130), (128, 127), (128, 70)])
@pytest.mark.parametrize("rows", [128, 640, 2176])
def test_attention_workspace_of_a_batch_serves_its_half(heads, most, rows):
    """129-255 (query, 64 heads) need none themselves; half as many split every list twice as often."""
    import torch
    from dsv41 import _abi
    size = lambda b: _abi.mla_workspace_bytes(b, 1, heads, 512, rows, torch.bfloat16)
    splits = 2                           # at least two splits per list: their bf16 numerators
    assert size(most) >= most * splits * heads * 512 * 2
    assert size(most // 2) > 0
    if rows >= 640:
        assert size(most) >= 0.98 * size(most // 2)
