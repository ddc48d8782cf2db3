"""The grouped output projection at chunk row counts, each tile shape against slices of decode row counts."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,groups,d,r", [
    (129, 8, 512, 1024), (256, 8, 64, 1024),     # 64 x 128 tiles
    (257, 8, 320, 1024), (511, 8, 512, 1024),    # 128 x 128, four stages; fewer steps than stages
    (513, 8, 512, 1024), (1279, 8, 128, 1024),   # 128 x 128, two per CU
    (1281, 8, 512, 1024), (1537, 8, 64, 1024),   # 256 x 256
    (700, 3, 256, 384), (6000, 3, 128, 384),     # widths that are no multiple of 256
])
def test_chunk_rows_equal_decode_rows(gpu, rows, groups, d, r):
    from dsv41 import _abi
    g = torch.Generator(device="cuda").manual_seed(rows)
    o = torch.randn(rows, groups * d, generator=g, device="cuda").bfloat16()
    w = torch.randn(groups * r, d, generator=g, device="cuda").bfloat16()
    got = _abi.wo_a_grouped(o, w, groups, out_dtype=torch.float32)
    few = torch.cat([_abi.wo_a_grouped(o[i:i + 128].contiguous(), w, groups, out_dtype=torch.float32)
                     for i in range(0, rows, 128)])
    assert torch.equal(got, few)
    assert torch.equal(_abi.wo_a_grouped(o, w, groups), few.bfloat16())


@pytest.mark.parametrize("rows", [1, 16, 17, 33])
def test_wide_projection_at_decode_rows(gpu, rows):
    """A projection of at least 16,384 outputs, on either side of the row count where the library takes over."""
    from dsv41.layers import decode_linear
    g = torch.Generator(device="cuda").manual_seed(rows)
    lin = torch.nn.Linear(192, 16384, bias=False, dtype=torch.bfloat16, device="cuda").requires_grad_(False)
    lin.weight.data.normal_(generator=g)
    x = torch.randn(rows, 192, generator=g, device="cuda").bfloat16()
    got = decode_linear(lin, x, wide_only=True)
    want = x.double() @ lin.weight.double().t()
    # one rounding to bf16 (2^-8 of the value) of a float32 sum of 192 exact products
    sums = 192 * 2 ** -23 * (x.double().abs() @ lin.weight.double().abs().t())
    assert ((got.double() - want).abs() <= want.abs() * 2 ** -8 + sums).all()


def test_wide_projection_keeps_what_the_module_call_does(gpu):
    """At decode rows the kernel stands in for lin(x): hooks, gradients, a forward of the module's own and
    tensors off 16-byte alignment still take the module."""
    from dsv41.layers import decode_linear
    lin = torch.nn.Linear(192, 16384, bias=False, dtype=torch.bfloat16, device="cuda").requires_grad_(False)
    x = torch.randn(4, 192, device="cuda").bfloat16()
    want = torch.nn.functional.linear(x, lin.weight)
    calls = []
    for register in (lin.register_forward_hook, lin.register_forward_pre_hook,
                     torch.nn.modules.module.register_module_forward_hook):
        handle = register(lambda *a: calls.append(a[0]))
        decode_linear(lin, x, wide_only=True)
        handle.remove()
    assert calls == [lin] * 3
    lin.forward = lambda t: torch.nn.functional.linear(t, lin.weight) * 2
    assert torch.equal(decode_linear(lin, x, wide_only=True), want * 2)
    del lin.forward

    off = torch.empty(x.numel() + 1, dtype=x.dtype, device="cuda")[1:].view_as(x).copy_(x)
    assert torch.equal(decode_linear(lin, off, wide_only=True), want)
    lin.weight = torch.nn.Parameter(torch.empty(lin.weight.numel() + 1, dtype=x.dtype, device="cuda")[1:].view(16384, 192)
                                    .copy_(lin.weight), requires_grad=False)
    assert lin.weight.data_ptr() % 16 and torch.equal(decode_linear(lin, x, wide_only=True), want)

    lin.requires_grad_(True)
    decode_linear(lin, x.requires_grad_(), wide_only=True).float().sum().backward()
    assert x.grad is not None and lin.weight.grad is not None


@pytest.mark.parametrize("k,n,rows,own", [(1280, 32768, 16, True), (1280, 32768, 17, False), (8192, 16384, 1, True),
                                          (4032, 32768, 16, True), (4096, 32768, 16, False), (1280, 65536, 12, False)])
def test_wide_projection_route(gpu, monkeypatch, k, n, rows, own):
    """Up to 16 rows the kernel takes outputs of 16,384 to 32,768; the library streams larger weights at least
    as fast."""
    from dsv41 import _abi, layers
    calls = []
    kernel = _abi.linear_rows
    monkeypatch.setattr(_abi, "linear_rows", lambda *a: calls.append(1) or kernel(*a))
    lin = torch.nn.Linear(k, n, bias=False, dtype=torch.bfloat16, device="cuda").requires_grad_(False)
    layers.decode_linear(lin, torch.randn(rows, k, device="cuda").bfloat16(), wide_only=True)
    assert bool(calls) == own
