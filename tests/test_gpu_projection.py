"""The projections' own kernels against float64: row counts around tiles and parts, widths that are not multiples of the
tiles, operands that are no ordinary numbers; and the calls that keep the library's operations."""
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


@pytest.mark.parametrize("N,K,O", [(1, 4, 2), (63, 36, 62), (64, 16, 64), (65, 20, 66), (130, 256, 130), (4097, 12, 128), (16385, 48, 256),
                                   (20001, 256, 258), (33000, 8, 64)])
@pytest.mark.parametrize("across", [False, True])
def test_product(N, K, O, across):
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(N + K + O)
    x, w, b = (torch.randn(*s, generator=g, device=dev) for s in ((N, K), (O, K), (O,)))
    assert projection._product_applies(N, O, K)
    got = projection._product(x, w.t().contiguous() if across else w, None if across else b, across)
    xd, wd, bd = x.double(), w.double(), torch.zeros_like(b).double() if across else b.double()
    # three parts hold all of a float32; what is left out is 2^-25 of a product at most, and each of K / 16 steps of six sums, and the bias,
    # is rounded (or cut) to 2^-23 of the running sum, at most the sum of the sizes
    bound = (2.0 ** -25 + (6 * (K // 16 + 1) + 16 + 1) * 2.0 ** -23) * (xd.abs() @ wd.abs().t() + bd.abs())
    assert ((got.double() - (xd @ wd.t() + bd)).abs() <= bound).all()
    again = projection._product(x, w.t().contiguous() if across else w, None if across else b, across)
    assert torch.equal(got, again)


def test_operands_that_are_no_ordinary_numbers():
    """Infinities, NaN, numbers that bfloat16 rounds to infinity, and tiny ones, whose parts are denormal: as the library's product."""
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    torch.manual_seed(1)
    x, w, b = torch.randn(4200, 64, device=dev), torch.randn(96, 64, device=dev), torch.randn(96, device=dev)
    w[:, 1] = 0.5
    x[3, 5], x[7, 9], x[200, 1], x[201, 1] = float("inf"), float("nan"), 3.402823e38, -3.402823e38
    x[50] *= 1e-34
    got, want = projection._product(x, w, b, False), torch.nn.functional.linear(x, w, b)
    torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-4, equal_nan=True)
    tiny = projection._product(x[50:51], w, None, False).double()
    torch.testing.assert_close(tiny, x[50:51].double() @ w.double().t(), rtol=0, atol=64 * 2.0 ** -23 * 1e-34 * 16)
    across = projection._product(x, w.t().contiguous(), None, True)
    torch.testing.assert_close(across, x.matmul(w.t()), rtol=1e-5, atol=1e-4, equal_nan=True)
    g = torch.randn(4200, 96, device=dev)
    g[9, 3], g[11, 6], x[11, 4], x[7, 9], x[3, 5] = float("inf"), 3.402823e38, 1.5, 0., 0.
    x[200:202] = 0
    gw, _ = projection._weight_gradients(x, g, True)
    torch.testing.assert_close(gw, g.t().mm(x), rtol=1e-4, atol=1e-2, equal_nan=True)


def test_offsets_keep_the_librarys_result_in_training():
    from dfa3D.modules.projection import Projection
    dev = torch.device("cuda:0")
    layer = Projection(256, 128, library_forward=True).to(dev)
    x = torch.randn(5000, 256, device=dev)
    assert torch.equal(layer(x), torch.nn.functional.linear(x, layer.weight, layer.bias))
    with torch.no_grad():
        torch.testing.assert_close(layer(x), torch.nn.functional.linear(x, layer.weight, layer.bias), rtol=1e-5, atol=1e-5)


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
