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


def test_compressor_shapes_outside_the_kernel(gpu):
    """Widths that are not whole tiles and float32 activations keep torch's linear."""
    from dsv41.compressor import _exact_weights_ok
    x, w0, w1 = _data(4, 96, 64, 64, 2)
    assert not _exact_weights_ok(x, w0, w1)
    x, w0, w1 = _data(4, 128, 128, 128, 2)
    assert _exact_weights_ok(x, w0, w1) and not _exact_weights_ok(x.float(), w0, w1)
