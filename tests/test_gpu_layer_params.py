"""GPU tests of the layers' one-launch parameter maps (``LayerParamsFn``) against
the torch operations they replace, in float64."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.gpu_util import announce, need_gpu

pytestmark = pytest.mark.gpu


def _inputs(n, seed):
    g = torch.Generator().manual_seed(seed)
    A = torch.randn(n, generator=g) * torch.rand(n, generator=g) * 40  # below, inside, above the band
    return A, torch.randn(n, generator=g), 3 * torch.randn(n, generator=g)


@pytest.mark.parametrize("damped", [True, False])
@pytest.mark.parametrize("n", [1, 127, 128, 129, 1000])
def test_layer_params_match_fp64(n, damped):
    """Values and gradients, elementwise.  The gradients are formed in double and
    rounded once: a few 2^-24."""
    need_gpu()
    from ossm_amd.layers import LayerParamsFn, project_parameters

    announce(f"layer params n={n} damped={damped}")
    A, G, s = _inputs(n, n)
    up = [torch.randn(n, generator=torch.Generator().manual_seed(i)) for i in range(3)]
    dev = [t.cuda().requires_grad_() for t in (A, G, s)]
    ref = [t.double().requires_grad_() for t in (A, G, s)]
    out = LayerParamsFn.apply(damped, dev[0], dev[1] if damped else None, dev[2])
    want = project_parameters(*ref) if damped else (torch.relu(ref[0]), 0 * ref[1], torch.sigmoid(ref[2]))
    lo, out = out[3], out[:3]
    if damped:  # the same float operations
        assert lo is None
        for o, w in zip(out, project_parameters(*dev)):
            assert torch.equal(o, w)
    else:  # value and residual together hold the double result to 2^-48
        assert not lo.requires_grad
        for o, w, l in zip(out, want, lo):
            np.testing.assert_allclose((o.detach().double() + l.double()).cpu().numpy(), w.detach().numpy(),
                                       rtol=2e-14, atol=1e-30)
    wrt = (0, 1, 2) if damped else (0, 2)
    got = torch.autograd.grad(out, [dev[i] for i in wrt], [u.cuda() for u in up])
    exp = torch.autograd.grad(want, [ref[i] for i in wrt], [u.double() for u in up])
    for x, r in zip(got, exp):
        np.testing.assert_allclose(x.cpu().numpy(), r.numpy(), rtol=1e-6,
                                   atol=1e-6 * float(r.abs().max()))
    # an output that nothing uses has no gradient
    a, g, dt, _ = LayerParamsFn.apply(damped, dev[0], dev[1] if damped else None, dev[2])
    only = torch.autograd.grad(dt, dev[2], up[2].cuda())[0]
    np.testing.assert_allclose(only.cpu().numpy(),
                               torch.autograd.grad(torch.sigmoid(ref[2]), ref[2], up[2].double())[0].numpy(),
                               rtol=1e-6, atol=1e-12)


def test_layer_params_pass_nan_and_differentiate_twice():
    need_gpu()
    from ossm_amd.layers import LayerParamsFn, project_parameters

    announce("layer params nan, create_graph")
    nan = torch.tensor([float("nan"), 1.0], device="cuda")
    one = torch.ones(2, device="cuda")
    assert torch.isnan(LayerParamsFn.apply(True, one, nan, one)[0][0])
    assert torch.isnan(LayerParamsFn.apply(False, nan, None, one)[0][0])
    A, G, s = (t.cuda().requires_grad_() for t in _inputs(17, 5))
    first = torch.autograd.grad(LayerParamsFn.apply(True, A, G, s)[0].square().sum(), s, create_graph=True)[0]
    second = torch.autograd.grad(first.sum(), s)[0]
    rA, rG, rs = (t.detach().double().requires_grad_() for t in (A, G, s))
    rf = torch.autograd.grad(project_parameters(rA, rG, rs)[0].square().sum(), rs, create_graph=True)[0]
    rsec = torch.autograd.grad(rf.sum(), rs)[0]
    # float32 torch operations on this path: lo loses about dt^2-scaled digits
    np.testing.assert_allclose(second.cpu().numpy(), rsec.cpu().numpy(), rtol=1e-3,
                               atol=1e-3 * float(rsec.abs().max()))


@pytest.mark.parametrize("disc", ["IM", "IMEX"])
@pytest.mark.parametrize("shape", [(2, 33, 1, 1), (1, 32, 256, 256), (3, 65, 40, 129)],
                         ids=lambda s: "x".join(map(str, s)))
def test_linoss_layer_fused_matches_composition(disc, shape, monkeypatch):
    """The LinOSS layer on the fused kernels against its composition of torch
    products and the scan (float32 both; each is within ~1e-5 of float64 here)."""
    need_gpu()
    from ossm_amd import linoss

    batch, length, hidden, ssm = shape
    torch.manual_seed(length + hidden)
    layer = linoss.LinOSSLayer(ssm, hidden, disc).cuda()
    u = torch.randn(batch, length, hidden, device="cuda", requires_grad=True)
    go = torch.randn(batch, length, hidden, device="cuda")
    announce(f"linoss layer fused {disc} {shape}")
    wrt = [u, *layer.parameters()]
    out = layer(u)
    got = [out, *torch.autograd.grad(out, wrt, go)]
    monkeypatch.setattr(linoss, "fused_layer_supported", lambda *a: False)
    out = layer(u)
    ref = [out, *torch.autograd.grad(out, wrt, go)]
    for x, r in zip(got, ref):
        x, r = x.detach().cpu().numpy(), r.detach().cpu().numpy()
        np.testing.assert_allclose(x, r, rtol=1e-4, atol=1e-4 * max(1.0, float(np.abs(r).max())))


@pytest.mark.parametrize("disc", ["IM", "IMEX"])
def test_layers_with_parameters_that_broadcast(disc):
    """Replaced parameters of one element are shared by all oscillators (channels), as
    by the torch operations; other sizes are refused."""
    need_gpu()
    from ossm_amd import layers, linoss

    announce(f"layers, broadcast parameters {disc}")
    torch.manual_seed(3)
    P = lambda v: torch.nn.Parameter(v.detach().clone())  # noqa: E731
    u = torch.randn(2, 40, 6, device="cuda")
    for make, shared in ((lambda: layers.DampedLinOSSLayer(7, 6), ("A_diag",)),
                         (lambda: linoss.LinOSSLayer(7, 6, disc), ("D", "steps") if disc == "IM" else ("D",))):
        torch.manual_seed(4)
        layer = make().cuda()
        for name in shared:
            p = getattr(layer, name)
            setattr(layer, name, P(p[:1].expand_as(p)))
        want = torch.autograd.grad(layer(u).square().sum(), [getattr(layer, n) for n in shared])
        for name in shared:
            setattr(layer, name, P(getattr(layer, name)[:1]))
        got = torch.autograd.grad(layer(u).square().sum(), [getattr(layer, n) for n in shared])
        for g, w in zip(got, want):
            np.testing.assert_allclose(g.cpu().numpy(), w.sum(0, keepdim=True).cpu().numpy(), rtol=1e-4, atol=1e-4)
        layer = make().cuda()
        layer.steps = torch.nn.Parameter(torch.zeros(9, device="cuda"))
        with pytest.raises(RuntimeError):
            layer(u)
