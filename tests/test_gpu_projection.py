"""The projections' own weight and bias gradient kernel against float64: row counts around its parts, widths that are not
multiples of its tiles; and the calls that keep the library's gradients."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(K, O, dev, seed=0):
    from dfa3D.modules.projection import Projection
    torch.manual_seed(seed)
    return Projection(K, O).to(dev)


@pytest.mark.parametrize("N,K,O", [(4096, 64, 64), (4097, 256, 512), (8191, 258, 66), (5000, 2, 2), (12345, 130, 254),
                                   (70001, 256, 256), (4111, 32, 640)])
def test_weight_and_bias_gradients(N, K, O):
    dev = torch.device("cuda:0")
    layer = _layer(K, O, dev)
    x = torch.randn(N, K, device=dev, requires_grad=True)
    g = torch.randn(N, O, device=dev)
    got = torch.autograd.grad(layer(x), [x, layer.weight, layer.bias], g)
    gd, xd = g.double().cpu(), x.detach().double().cpu()
    want = (gd @ layer.weight.detach().double().cpu(), gd.t() @ xd, gd.sum(0))
    # sums of N products of unit variance in float32: N^(1/2) in size, rounded to 2^-24 of the running sum at most N^(1/2)
    # times with random signs, so 1e-6 of the largest partial sum (about 4 N^(1/2)) leaves an order of magnitude
    for a, b, n in zip(got, want, (O, N, N)):
        assert (a.double().cpu() - b).abs().max() <= 4e-6 * n ** 0.5 * 4
    again = torch.autograd.grad(layer(x), [layer.weight, layer.bias], g)
    assert torch.equal(again[0], got[1]) and torch.equal(again[1], got[2])      # fixed order of summation


def test_rows_in_other_layouts_and_partial_gradients():
    """Three-dimensional input, a gradient that is not contiguous, only some of the gradients asked for."""
    dev = torch.device("cuda:0")
    layer = _layer(64, 96, dev)
    x = torch.randn(5000, 3, 64, device=dev).transpose(0, 1)
    g = torch.randn(96, 3, 5000, device=dev).permute(1, 2, 0)
    want_w, want_b = torch.einsum("abo,abk->ok", g.double().cpu(), x.double().cpu()), g.double().cpu().sum((0, 1))
    gw, gb = torch.autograd.grad(layer(x), [layer.weight, layer.bias], g)
    torch.testing.assert_close(gw.double().cpu(), want_w, rtol=0, atol=2e-3)
    torch.testing.assert_close(gb.double().cpu(), want_b, rtol=0, atol=2e-3)
    gw2, = torch.autograd.grad(layer(x), [layer.weight], g)
    assert torch.equal(gw2, gw)


def test_calls_that_keep_the_librarys_operation():
    """Second derivatives, functorch transforms, forward-mode derivatives, autocast and few rows."""
    dev = torch.device("cuda:0")
    layer = _layer(64, 64, dev)
    x = torch.randn(4200, 64, device=dev, requires_grad=True)
    gw, = torch.autograd.grad(layer(x).square().sum(), [layer.weight], create_graph=True)
    second, = torch.autograd.grad(gw.square().sum(), [x])
    ref = torch.nn.functional.linear
    rw, = torch.autograd.grad(ref(x, layer.weight, layer.bias).square().sum(), [layer.weight], create_graph=True)
    want, = torch.autograd.grad(rw.square().sum(), [x])
    torch.testing.assert_close(second, want, rtol=1e-3, atol=1e-3 * want.abs().max().item())
    gs = torch.randn(3, 4200, 64, device=dev)
    batched, = torch.autograd.grad(layer(x), [layer.weight], gs, is_grads_batched=True)
    torch.testing.assert_close(batched, gs.transpose(1, 2) @ x.detach(), rtol=1e-3, atol=1e-2)
    per = torch.func.vmap(lambda t: layer(t))(x.detach().view(1, 4200, 64))
    torch.testing.assert_close(per[0], layer(x.detach()))
    out, tangent = torch.func.jvp(lambda t: layer(t), (x.detach(),), (torch.ones_like(x),))
    torch.testing.assert_close(tangent, torch.ones_like(x) @ layer.weight.detach().t(), rtol=1e-4, atol=1e-4)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert layer(x).dtype == torch.bfloat16
    few = torch.randn(7, 64, device=dev)
    torch.autograd.grad(layer(few).sum(), [layer.weight])
