"""Selection over many rows (a chunk's queries) against the same rows selected a few at a time, which take other kernels."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _scores(rows, nb, kind):
    g = torch.Generator(device="cuda").manual_seed(rows + nb)
    x = torch.randn(rows, 1, nb, generator=g, device="cuda")
    if kind == "ties":                   # five values, both zeros among them
        x = (x * 1.2).round().clamp(-2, 2)
        x = torch.where(x == 0, torch.where(torch.rand(x.shape, generator=g, device="cuda") < 0.5, -0.0, 0.0), x)
    elif kind == "masked":               # most entries -inf, some rows with fewer finite ones than k
        x.masked_fill_(torch.rand(x.shape, generator=g, device="cuda") < 0.97, -float("inf"))
        x[:3] = -float("inf")
    elif kind == "odd":                  # infinities and NaNs of both signs, the all-ones one included
        bits = x.view(torch.int32)
        pick = torch.randint(0, 12, x.shape, generator=g, device="cuda")
        for i, v in enumerate((0x7F800000, -0x800000, 0x7FC00000, -0x400000, -1)):
            bits.masked_fill_(pick == i, v)
    return x.contiguous()


@pytest.mark.parametrize("rows,nb,k", [
    (512, 2, 1), (513, 65, 64), (512, 2048, 512), (600, 2049, 2048), (512, 4096, 1), (512, 4097, 512),
    (512, 6145, 6144), (512, 8193, 777), (530, 10240, 2048), (512, 10241, 512), (512, 12289, 512), (512, 16384, 1024),
    (64, 16385, 512), (70, 20481, 2048), (64, 24577, 512), (64, 32768, 4096),
    (79, 24577, 1024), (80, 24577, 1024), (64, 32768, 1025),
    (128, 32769, 512),                   # two chunks, the second a little shorter
    (130, 65536, 2048), (128, 65600, 512),
    (128, 98305, 4096),                  # four chunks
])
@pytest.mark.parametrize("kind", ["normal", "ties", "masked", "odd"])
def test_rows_equal_few_rows(gpu, rows, nb, k, kind):
    from dsv41 import _abi
    x = _scores(rows, nb, kind)
    start = nb - nb // 7                 # the last positions are past the queries' visibility
    got = _abi.topk_select(x, k, start, 1, 5)
    few = torch.cat([_abi.topk_select(x[i:i + 31].contiguous(), k, start, 1, 5) for i in range(0, rows, 31)])
    assert torch.equal(got, few)


@pytest.mark.parametrize("nb,k", [(2048, 600), (10240, 2048), (32768, 512)])
@pytest.mark.parametrize("inf", [0.0, 0.02, 0.5])
def test_rows_down_to_infinity_and_below(gpu, nb, k, inf):
    """The k-th best is -inf, or a NaN below it: entries the first histogram leaves out."""
    from dsv41 import _abi
    g = torch.Generator(device="cuda").manual_seed(nb)
    x = torch.full((512, 1, nb), -float("nan"), device="cuda")
    x.view(torch.int32).masked_fill_(torch.rand(x.shape, generator=g, device="cuda") < 0.3, -1)
    x.masked_fill_(torch.rand(x.shape, generator=g, device="cuda") < inf, -float("inf"))
    x[:, :, 5:20] = 1.0
    x.view(torch.int32)[100:200, :, 20:] = -0x400000       # rows of equal NaNs
    got = _abi.topk_select(x, k, nb, 1, 0)
    few = torch.cat([_abi.topk_select(x[i:i + 31].contiguous(), k, nb, 1, 0) for i in range(0, 512, 31)])
    assert torch.equal(got, few)


@pytest.mark.parametrize("rows,nb,kb", [
    (512, 9, 1), (512, 4097, 300), (513, 16384, 2047), (520, 16385, 2048), (515, 22804, 2048),
    (512, 32776, 4096), (512, 65536, 1),
    (64, 8193, 700), (383, 8192, 64), (384, 8192, 64),   # either side of 1,024 blocks and of 384 rows
])
@pytest.mark.parametrize("kind", ["normal", "ties", "masked", "odd"])
def test_candidate_rows_equal_few_rows(gpu, rows, nb, kb, kind):
    """Candidate blocks of many rows, 8 scores a block, against the same rows a few at a time."""
    from dsv41 import _abi
    x = _scores(rows, nb, kind)
    x[7] = float("nan")                  # blocks of nothing but NaN
    x[8, :, :64] = -float("nan")
    lens = torch.tensor([nb - nb // 7], dtype=torch.int32, device="cuda")
    got = _abi.candidate_blocks(x, kb, 8, lens)
    few = torch.cat([_abi.candidate_blocks(x[i:i + 63].contiguous(), kb, 8, lens) for i in range(0, rows, 63)])
    assert torch.equal(got, few)


@pytest.mark.parametrize("nb,kb,past", [(1999, 100, 1), (1999, 100, 40), (4104, 64, 8), (16384, 2047, 300)])
def test_candidate_rows_visible_past_their_end(gpu, nb, kb, past):
    """A visibility beyond the row pins no block: all kb places go to the row's own blocks."""
    from dsv41 import _abi
    x = _scores(520, nb, "normal")
    lens = torch.tensor([nb + past], dtype=torch.int32, device="cuda")
    got = _abi.candidate_blocks(x, kb, 8, lens)
    few = torch.cat([_abi.candidate_blocks(x[i:i + 63].contiguous(), kb, 8, lens) for i in range(0, 520, 63)])
    assert torch.equal(got, few)
    pad = torch.nn.functional.pad(got, (0, -nb % 8)).unflatten(-1, (-1, 8))
    assert bool((pad.any(-1).sum(-1) == kb).all())


def test_rows_of_several_queries(gpu):
    """Visibility follows the query, row % n, also with rows of several sequences and k >= nb."""
    from dsv41 import _abi
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(3, 211, 900, generator=g, device="cuda")
    for k in (100, 900, 2000):
        got = _abi.topk_select(x, k, 700, 2, 9)
        few = torch.cat([_abi.topk_select(x[:, i:i + 1].contiguous(), k, 700 + i, 2, 9) for i in range(211)], 1)
        assert torch.equal(got, few)


def _select_ws(x, k, ws):
    from dsv41 import _abi
    rows, _, nb = x.shape
    out = torch.empty(rows, 1, k, dtype=torch.int32, device="cuda")
    _abi._call("dsv41_topk_select_ws", _abi._ptr(x), _abi._ptr(out), rows, 1, nb, k, 2 * nb, 1, 0, _abi._ptr(ws),
               ws.numel() if ws is not None else 0, _abi._stream(x))
    return out


def test_workspace_matches_the_route(gpu):
    """Two-stage rows state their workspace and refuse less than they use."""
    from dsv41 import _abi
    used = 2 * 128 * 2 * 512 * 4         # two chunks' lists of 512 keys and positions
    assert _abi.topk_workspace_bytes(128, 65536, 512) >= used
    x = torch.randn(128, 1, 65536, device="cuda")
    small = torch.empty(used - 256, dtype=torch.uint8, device="cuda")
    with pytest.raises(ValueError):
        _select_ws(x, 512, small)


@pytest.mark.parametrize("nb,k,most,fewer", [(32768, 512, 64, (63, 64, 31)), (32768, 512, 2048, (63, 600)),
                                             (65536, 512, 128, (127, 128, 5)), (20001, 1024, 300, (63, 64, 300))])
def test_workspace_of_the_most_rows_serves_fewer(gpu, nb, k, most, fewer):
    from dsv41 import _abi
    ws = torch.empty(_abi.topk_workspace_bytes(most, nb, k), dtype=torch.uint8, device="cuda")
    x = _scores(max(fewer), nb, "normal")
    for rows in fewer:
        part = x[:rows].contiguous()
        assert torch.equal(_select_ws(part, k, ws), _abi.topk_select(part, k, 2 * nb, 1, 0))


def test_many_rows_without_a_workspace(gpu):
    """k over half a chunk: few rows take one stage and no workspace, many take two only if they get one."""
    from dsv41 import _abi
    assert _abi.topk_workspace_bytes(127, 65536, 3000) == 0 < _abi.topk_workspace_bytes(128, 65536, 3000)
    x = _scores(128, 65536, "ties")
    assert torch.equal(_select_ws(x, 3000, None), _abi.topk_select(x, 3000, 131072, 1, 0))
