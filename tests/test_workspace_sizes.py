"""Workspace sizes are host arithmetic: one sized for the largest batch has to serve every smaller one."""

from __future__ import annotations

import pytest


@pytest.mark.parametrize("nb,k", [(16385, 512), (20000, 1024), (32768, 512), (32768, 2048), (32769, 512),
                                  (65536, 512), (65536, 3000), (131072, 1024), (400000, 64)])
def test_topk_workspace_never_falls_with_rows(nb, k):
    from dsv41 import _abi
    sizes = [_abi.topk_workspace_bytes(r, nb, k) for r in list(range(1, 700)) + [2048, 8192, 65536]]
    assert sizes == sorted(sizes)
