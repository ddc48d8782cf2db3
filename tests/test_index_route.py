"""Which chunks under a candidate mask take the fused scoring and selection: host arithmetic, on the CPU."""

from __future__ import annotations

import pytest


@pytest.mark.parametrize("queries,nb,topk,mxfp4,two", [
    (8, 8192, 512, False, True), (8, 8193, 512, False, False), (8, 8192, 128, True, True),
    (64, 12288, 512, False, True), (63, 12288, 512, False, False), (64, 12288, 128, True, True),
    (8, 32768, 512, False, False), (8, 32769, 512, False, True), (8, 32769, 511, False, False),
    (64, 32764, 512, True, False), (64, 32764, 1024, True, True), (64, 32764, 512, False, True),
    (64, 24576, 512, True, True), (96, 32768, 512, True, True), (2048, 32768, 512, True, True),
])
def test_two_calls(queries, nb, topk, mxfp4, two):
    from dsv41.indexer import _score_then_select
    assert _score_then_select(queries, nb, topk, mxfp4) == two


def test_short_chunks_and_masks():
    """Fewer than 8 queries per sequence are asked of the fused form, chunks without a mask are not."""
    from types import SimpleNamespace
    from dsv41.indexer import Indexer
    layer = SimpleNamespace(n_heads=32, index_topk=512)
    assert Indexer._fused(layer, 16, 7, 16384, None) and Indexer._fused(layer, 16, 7, 16384, object())
    assert not Indexer._fused(layer, 1, 8, 16384, None)
    assert Indexer._fused(layer, 1, 8, 16384, object()) and not Indexer._fused(layer, 1, 2048, 16384, object())
