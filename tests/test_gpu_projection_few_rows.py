"""Training calls of the projections with few rows, which the library formed before: a single row, rows around the tiles, sums of several layers' terms
whatever their depth; and no rows at all."""
import pytest
import torch

from dfa3D.modules import projection
from dfa3D.modules.projection import Projection, projections

pytestmark = pytest.mark.gpu


def _error(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("N", [1, 5, 64, 129, 1000, 4095])
@pytest.mark.parametrize("widths", [(256,), (512, 256, 256), (66, 64), (2, 4, 130, 8)])
def test_gradients(N, widths):
    """No further from float64 than the library's, of which each sum of n terms is within n 2^-24 of the sum of their sizes."""
    dev, K = torch.device("cuda:0"), 256
    torch.manual_seed(N + sum(widths))
    layers = [Projection(K, O, library_forward=i == 0).to(dev) for i, O in enumerate(widths)]
    x = torch.randn(2, N, K, device=dev, requires_grad=True)
    gs = [torch.randn(2, N, O, device=dev) for O in widths]
    params = [p for l in layers for p in (l.weight, l.bias)]
    out = projections(x, layers)
    assert "Function" in out[0].grad_fn.name() and torch.equal(out[0], torch.nn.functional.linear(x, layers[0].weight, layers[0].bias))
    grads = torch.autograd.grad(out, [x] + params, gs)
    rows, flat = x.detach().reshape(-1, K), [g.reshape(-1, g.shape[-1]) for g in gs]
    want = sum(g.double() @ l.weight.detach().double() for g, l in zip(flat, layers)).view_as(x)
    library = sum(g @ l.weight.detach() for g, l in zip(gs, layers))
    assert _error(grads[0], want) <= 1.1 * _error(library, want) + 1e-7
    for i, g in enumerate(flat):
        want = g.double().t() @ rows.double()
        assert _error(grads[1 + 2 * i], want) <= 1.1 * _error(g.t().mm(rows), want) + 1e-7
        assert _error(grads[2 + 2 * i], g.double().sum(0)) <= 5e-7
    again = torch.autograd.grad(projections(x, layers), [x] + params, gs)
    assert all(torch.equal(a, b) for a, b in zip(again, grads))                # fixed order of summation


def test_no_rows():
    dev = torch.device("cuda:0")
    layer = Projection(16, 8).to(dev)
    x = torch.randn(0, 16, device=dev, requires_grad=True)
    gx, gw = torch.autograd.grad(layer(x).sum(), [x, layer.weight])
    assert gx.shape == x.shape and not gw.any()


def test_deep_sums_of_several_layers_only():
    """Up to 1024 terms of several layers; one deep layer, and more terms, with few rows stay with the library."""
    dev = torch.device("cuda:0")
    pairs = lambda *widths: tuple(t for O in widths for t in (torch.randn(100, O, device=dev), torch.randn(O, 256, device=dev)))
    assert projection._sum_of_products(pairs(512, 512)) is not None
    assert projection._sum_of_products(pairs(512)) is None and projection._sum_of_products(pairs(512, 516)) is None
    assert projection._sum_of_products(pairs(510, 4)) is None                  # widths of whole groups of four
