"""GPU tests of ``rows_product`` (weight gradients on the split-bf16 matrix-core
kernel) and of the projections that use it."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.gpu_util import announce, need_gpu

pytestmark = pytest.mark.gpu


def _bound(a, b):
    """|error| of a float32 product sum_r a b, split terms dropped at 2^-25 and
    summed in runs of 16: a few 2^-24 of sum |a b| covers both."""
    return 4 * 2.0 ** -24 * (a.abs().double().t() @ b.abs().double())


# one block, a last block of one row, a ragged last block, tiles with one
# column, exact tiles, columns past a tile, more tiles than CUs / slices
@pytest.mark.parametrize("shape", [(16, 3, 2), (17, 130, 66), (512, 1, 1), (513, 128, 64), (527, 129, 65), (1000, 4, 130), (4097, 36, 128),
                                   (20000, 256, 3), (640, 2050, 1030)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("layout", ["plain", "pairs", "strided", "odd_stride"])
def test_rows_product_against_float64(shape, layout):
    need_gpu()
    from ossm_amd.linear import rows_product

    R, M, N = shape
    if layout == "pairs" and M % 2:
        M += 1
    announce(f"rows_product {R}x{M}x{N} {layout}")
    g = torch.Generator().manual_seed(R + M)
    pad = {"plain": 0, "pairs": 0, "strided": 8, "odd_stride": 3}[layout]
    a = (torch.randn(R, M + pad, generator=g) * torch.exp(torch.randn(R, 1, generator=g))).cuda()
    b = torch.randn(R, N + pad, generator=g).cuda()
    a, b = a[:, pad:], b[:, :N]
    got = rows_product(a, b, pairs=layout == "pairs")
    want = a.double().t() @ b.double()
    bound = _bound(a, b)
    if layout == "pairs":
        want, bound = (t.reshape(M // 2, 2, N).transpose(1, 2) for t in (want, bound))
    assert got.shape == want.shape and got.is_contiguous()
    assert bool(((got.double() - want).abs() <= bound).all())
    assert torch.equal(got, rows_product(a, b, pairs=layout == "pairs"))  # fixed order


def test_rows_product_wide_range_and_special_values():
    """Magnitudes down to the split's last term, exact powers, a NaN column and an
    infinity (NaN or infinity where float32 has one; other columns untouched)."""
    need_gpu()
    from ossm_amd.linear import rows_product

    announce("rows_product special values")
    a = torch.randn(600, 8, device="cuda") * torch.logspace(-30, 30, 8, device="cuda")
    b = torch.randn(600, 6, device="cuda")
    got, want = rows_product(a, b), a.double().t() @ b.double()
    assert bool(((got.double() - want).abs() <= _bound(a, b)).all())
    a[3, 2], a[5, 4] = float("nan"), float("inf")
    got = rows_product(a, b)
    bad = ~torch.isfinite(got)
    assert bool(bad[2].all()) and bool(bad[4].all()) and not bool(bad[[0, 1, 3, 5, 6, 7]].any())


def test_rows_product_infinities_and_largest_values():
    """Infinite and overflowing sums are infinities of float32's sign, and values past
    bfloat16's largest, which rounds to infinity, are values (several row counts: a
    wave's only block, its last one, one of many)."""
    need_gpu()
    from ossm_amd.linear import rows_product

    for R in (16, 640, 70000):
        announce(f"rows_product infinities R={R}")
        a, b = torch.randn(R, 130, device="cuda"), torch.randn(R, 67, device="cuda")
        a[R - 3, 4], b[7, 66] = float("inf"), -float("inf")
        a[R // 2, 129] = torch.finfo(torch.float32).max
        b[R // 2] *= 2.0 ** -20
        a[9, 64], b[9, 3] = 1e30, 1e30
        # the sum of (inf, -inf) and of NaN with anything are NaN both ways
        got, want = rows_product(a, b), (a.double().t() @ b.double()).float()
        assert torch.equal(torch.isfinite(got), torch.isfinite(want))
        bad = ~torch.isfinite(want)
        assert torch.equal(got[bad].nan_to_num(0.0), want[bad].nan_to_num(0.0))
        bound = torch.where(bad, 0.0, _bound(a, b))
        assert bool(((got.double() - want.double()).abs()[~bad] <= bound[~bad]).all())


@pytest.mark.parametrize("bias", [True, False])
def test_linear_matches_module(bias):
    """Outputs, and gradients of x, weight and bias, against the module's own; a
    hooked, replaced or small module is called as it is; create_graph works."""
    need_gpu()
    from ossm_amd.linear import linear

    announce(f"linear bias={bias}")
    torch.manual_seed(3)
    m = torch.nn.Linear(40, 24, bias=bias).cuda()
    x = torch.randn(5, 200, 40, device="cuda", requires_grad=True)
    go = torch.randn(5, 200, 24, device="cuda")
    y = linear(m, x)
    assert "LinearFn" in type(y.grad_fn).__name__ and torch.equal(y, m(x))
    wrt = [x, *m.parameters()]
    for g, r in zip(torch.autograd.grad(y, wrt, go), torch.autograd.grad(m(x), wrt, go)):
        np.testing.assert_allclose(g.cpu().numpy(), r.cpu().numpy(), rtol=1e-4, atol=1e-4)
    gw = torch.autograd.grad(linear(m, x).square().sum(), m.weight, create_graph=True)[0]
    ref = torch.autograd.grad(m(x).square().sum(), m.weight, create_graph=True)[0]
    for g, r in zip(torch.autograd.grad(gw.sum(), wrt, allow_unused=True),
                    torch.autograd.grad(ref.sum(), wrt, allow_unused=True)):
        np.testing.assert_allclose(g.cpu().numpy(), r.cpu().numpy(), rtol=1e-4, atol=1e-2)
    calls = []
    handle = m.register_forward_hook(lambda *a: calls.append(1))
    linear(m, x)
    handle.remove()
    assert calls == [1]
    assert "LinearFn" not in type(linear(m, x[:, :3]).grad_fn).__name__
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert linear(m, x).dtype == torch.bfloat16
