"""The compressor's float32 projections on the bf16 matrix cores against float64."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _data(rows, k, n0, n1, seed, spread=0.0):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rnd(*shape):
        x = torch.randn(*shape, generator=g, device="cuda")
        return x * torch.exp2(spread * torch.randn(*shape, generator=g, device="cuda").round()) if spread else x

    return rnd(rows, k).bfloat16(), rnd(n0, k) * 0.02, rnd(n1, k) * 0.02


@pytest.mark.parametrize("rows,k,n0,n1,spread", [
    (1, 64, 128, 128, 0),                # one 64-channel step, one range
    (31, 5120, 512, 512, 0), (33, 5120, 512, 512, 0), (65, 1024, 256, 128, 0),
    (129, 5120, 512, 512, 0), (1023, 192, 128, 384, 0), (1025, 5120, 512, 512, 0),
    (4097, 640, 512, 512, 0),            # the largest tiles, a last tile of one row
    (200, 320, 128, 128, 8.0),           # weights and activations over 2**-24 .. 2**24
])
def test_projections_against_float64(gpu, rows, k, n0, n1, spread):
    from dsv41 import _abi
    x, w0, w1 = _data(rows, k, n0, n1, rows + k, spread)
    for y, w in zip(_abi.linear_f32_pair(x, w0, w1), (w0, w1)):
        exact = x.double() @ w.double().t()
        mass = x.double().abs() @ w.double().abs().t()
        # exact products; at most one float32 rounding per MFMA (three per 32 channels) and per range
        bound = (3 * k / 32 + 40) * 2.0 ** -24 * mass
        assert y.dtype == torch.float32 and bool(((y.double() - exact).abs() <= bound).all())
        off = (y.double() - exact).norm()
        if spread:
            # one product dominates each sum: its three partial products are rounded into the sum one
            # after another, at most 2**-24 of the result each
            assert off <= 3 * 2.0 ** -24 * exact.norm()
        else:
            assert off <= 1.05 * (F.linear(x.float(), w).double() - exact).norm()


def test_projections_with_infinities(gpu):
    """Infinite activations and weights, with exactly representable weights (whose lower planes are 0)."""
    from dsv41 import _abi
    x, w0, w1 = _data(70, 128, 128, 128, 9)
    w0 = w0.sign()
    x[3, 5], x[4, 6], x[5, 7] = float("inf"), float("-inf"), float("nan")
    w1[2, 9], w1[7, 11] = float("inf"), float("nan")
    for y, w in zip(_abi.linear_f32_pair(x, w0, w1), (w0, w1)):
        lib = F.linear(x.float(), w)
        assert torch.equal(y.isnan(), lib.isnan())
        assert torch.equal(y[y.isinf()], lib[lib.isinf()])


@pytest.mark.parametrize("rows,k", [(5, 5120), (70, 320), (300, 192), (1025, 448), (4097, 128)])
def test_infinities_in_every_tile(gpu, rows, k):
    """Infinite and NaN activations and weights against float64, per tile size and with ranges; every output
    they do not reach keeps its bits."""
    from dsv41 import _abi
    x, w0, w1 = _data(rows, k, 128, 128, rows)
    clean = _abi.linear_f32_pair(x, w0, w1)
    x[0, 3], x[1, 70 % k], x[2, 9] = float("inf"), float("-inf"), float("nan")
    x[rows - 1, 5], x[rows - 1, k - 1] = float("inf"), float("-inf")
    w0[3, 11], w0[127, k - 2] = float("-inf"), float("inf")
    w1[64, 20] = float("nan")
    w1[5, 3], w1[6, 3], w1[7, 3] = 0.0, 1e-41, -1e-41       # times the infinite activation: NaN, inf, -inf
    hit = x.float().isfinite().all(1, keepdim=True)
    for y, w, c in zip(_abi.linear_f32_pair(x, w0, w1), (w0, w1), clean):
        want = x.double() @ w.double().t()
        assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isposinf(), want.isposinf())
        assert torch.equal(y.isneginf(), want.isneginf())
        keep = hit & w.isfinite().all(1) & (torch.arange(128, device="cuda") > 7)
        assert torch.equal(y[keep], c[keep])


@pytest.mark.parametrize("rows", [64, 2000])
def test_nan_rows_take_a_few_times_as_long_at_most(gpu, rows):
    """A poisoned batch must not hold up the launch: one re-evaluation on the matrix cores (measured 2 to 5
    times the finite time; the bound leaves room for a busy card)."""
    from dsv41 import _abi

    def best_us(x):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        us = []
        for _ in range(5):
            e[0].record()
            y = _abi.linear_f32_pair(x, w0, w1)
            e[1].record()
            torch.cuda.synchronize()
            us.append(e[0].elapsed_time(e[1]) * 1e3)
        return min(us), y[0]

    x, w0, w1 = _data(rows, 5120, 512, 512, 1)
    finite, _ = best_us(x)
    poisoned, y = best_us(torch.full_like(x, float("nan")))
    assert bool(y.isnan().all()) and poisoned < 20 * finite + 50


def test_compressor_shapes_outside_the_kernel(gpu):
    """Widths that are not whole tiles and float32 activations keep torch's linear."""
    from dsv41.compressor import _exact_weights_ok
    x, w0, w1 = _data(4, 96, 64, 64, 2)
    assert not _exact_weights_ok(x, w0, w1)
    x, w0, w1 = _data(4, 128, 128, 128, 2)
    assert _exact_weights_ok(x, w0, w1) and not _exact_weights_ok(x.float(), w0, w1)


@pytest.mark.parametrize("b,n,start,ratio,k", [
    (1, 1, 1, 2, 64),                    # one token closes a group; one contraction range
    (32, 1, 4095, 4, 5120), (3, 1, 4094, 4, 5120),       # the second leaves its group open
    (1, 300, 401, 2, 5120), (2, 77, 6, 4, 1024), (5, 3, 0, 4, 320),
    (1, 1025, 7, 4, 640), (1, 4099, 2, 4, 128),          # one range at the last size: no parts
])
def test_chunk_equals_projections_and_pool(gpu, b, n, start, ratio, k):
    from dsv41 import _abi
    x, w0, w1 = _data(b * n, k, 512, 512, n + k)
    x = x.view(b, n, k)
    if n == 77:
        x[1, 3, 5], x[0, 9, 2] = float("inf"), float("nan")
        w1[7, 3] = float("-inf")
    g = torch.Generator(device="cuda").manual_seed(n)
    st = [torch.randn(b + 1, ratio, 512, generator=g, device="cuda") for _ in range(2)]
    st2 = [t.clone() for t in st]
    norm = torch.rand(512, generator=g, device="cuda") + 0.5
    kv, score = _abi.linear_f32_pair(x, w0, w1)
    want = _abi.compress_pool(kv, score, *st, norm, ratio, start, 1e-6, torch.bfloat16)
    got = _abi.compress_chunk(x, w0, w1, *st2, norm, ratio, start, 1e-6)
    assert (want is None) == (got is None)
    for a, c in zip(([] if want is None else [want]) + st, ([] if got is None else [got]) + st2):
        assert torch.equal(a.isnan(), c.isnan())
        assert torch.equal(a.nan_to_num(7.0), c.nan_to_num(7.0))


@pytest.mark.parametrize("rows,k", [(129, 320), (700, 832), (1300, 448), (2500, 5120), (5000, 1088)])
def test_ranges_of_unequal_length(gpu, rows, k):
    """Row counts whose ranges do not divide the contraction's steps evenly."""
    from dsv41 import _abi
    x, w0, w1 = _data(rows, k, 512, 512, rows)
    for y, w in zip(_abi.linear_f32_pair(x, w0, w1), (w0, w1)):
        exact = x.double() @ w.double().t()
        bound = (3 * k / 32 + 40) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())   # as above
        assert bool(((y.double() - exact).abs() <= bound).all())
        assert (y.double() - exact).norm() <= 1.05 * (F.linear(x.float(), w).double() - exact).norm()
