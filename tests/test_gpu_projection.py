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


@pytest.mark.parametrize("N,K,O", [(1, 4, 4), (63, 36, 64), (64, 16, 64), (65, 20, 68), (130, 256, 132), (4097, 12, 128), (16385, 48, 256),
                                   (20001, 256, 260), (33000, 8, 64)])
@pytest.mark.parametrize("across", [False, True])
def test_product(N, K, O, across):
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(N + K + O)
    x, w, b = (torch.randn(*s, generator=g, device=dev) for s in ((N, K), (O, K), (O,)))
    product = lambda: projection._sum_of_products((x, w.t().contiguous())) if across else projection._product(x, w, b)
    got = product()
    xd, wd, bd = x.double(), w.double(), torch.zeros_like(b).double() if across else b.double()
    # three parts hold all of a float32; what is left out is 2^-25 of a product at most, and each of K / 16 steps of six sums, and the bias,
    # is rounded (or cut) to 2^-23 of the running sum, at most the sum of the sizes
    bound = (2.0 ** -25 + (6 * (K // 16 + 1) + 16 + 1) * 2.0 ** -23) * (xd.abs() @ wd.abs().t() + bd.abs())
    assert ((got.double() - (xd @ wd.t() + bd)).abs() <= bound).all()
    assert torch.equal(got, product())


def test_operands_that_are_no_ordinary_numbers():
    """Infinities, NaN, numbers that bfloat16 rounds to infinity, and tiny ones, whose parts are denormal: as the library's product."""
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    torch.manual_seed(1)
    x, w, b = torch.randn(4200, 64, device=dev), torch.randn(96, 64, device=dev), torch.randn(96, device=dev)
    w[:, 1] = 0.5
    x[3, 5], x[7, 9], x[200, 1], x[201, 1] = float("inf"), float("nan"), 3.402823e38, -3.402823e38
    x[50] *= 1e-34
    got, want = projection._product(x, w, b), torch.nn.functional.linear(x, w, b)
    torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-4, equal_nan=True)
    tiny = projection._product(x[50:51], w, None).double()
    torch.testing.assert_close(tiny, x[50:51].double() @ w.double().t(), rtol=0, atol=64 * 2.0 ** -23 * 1e-34 * 16)
    across = projection._sum_of_products((x, w.t().contiguous()))
    torch.testing.assert_close(across, x.matmul(w.t()), rtol=1e-5, atol=1e-4, equal_nan=True)
    g = torch.randn(4200, 96, device=dev)
    g[9, 3], g[11, 6], x[11, 4], x[7, 9], x[3, 5] = float("inf"), 3.402823e38, 1.5, 0., 0.
    x[200:202] = 0
    gw, _ = projection._weight_gradients(x, g, True)
    torch.testing.assert_close(gw, g.t().mm(x), rtol=1e-4, atol=1e-2, equal_nan=True)


# on both sides of the lines that the launcher draws: one tile of 32 rows per workgroup, two, three, five and nine, of one block of 256 columns, two and three
@pytest.mark.parametrize("N,K,O", [(4928, 256, 130), (8192, 256, 256), (12289, 196, 256), (12320, 252, 258), (24607, 256, 512), (50000, 256, 160),
                                   (5001, 252, 250), (12300, 228, 254), (16411, 196, 200), (16500, 228, 506), (25003, 256, 642), (25003, 252, 706), (32801, 200, 130),
                                   (33000, 256, 386), (33000, 196, 450), (65600, 196, 196), (65600, 212, 324), (65600, 200, 258)])
@pytest.mark.parametrize("across", [False, True])
def test_product_with_the_weight_in_registers(N, K, O, across):
    """Row tiles that end early, one tile per workgroup and several, depths and widths that are no whole steps or columns of a wavefront; rows with
    an infinity, a NaN, huge and tiny numbers in the first, a middle and the last tile, next to rows without."""
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(N + K + O)
    x, w, b = (torch.randn(*s, generator=g, device=dev) for s in ((N, K), (O, K), (O,)))
    wt = w.t().contiguous()
    product = lambda: projection._sum_of_products((x, wt)) if across else projection._product(x, w, b)
    want = x.double() @ w.double().t() + (0 if across else b.double())
    bound = (2.0 ** -25 + (6 * (K // 16 + 1) + 16 + 1) * 2.0 ** -23) * (x.double().abs() @ w.double().abs().t() + b.double().abs())      # as in test_product
    got = product()
    assert ((got.double() - want).abs() <= bound).all()
    assert torch.equal(got, product())
    odd = torch.tensor([3, N // 2, N // 2 + 33, N - 1], device=dev)
    x[odd[0], 5], x[odd[1], K - 1], x[odd[2], 0] = float("inf"), float("nan"), 3e38
    x[odd[3]] *= 1e-34
    again = product()
    library = x[odd] @ wt if across else torch.nn.functional.linear(x[odd], w, b)
    torch.testing.assert_close(again[odd[:3]], library[:3], rtol=1e-5, atol=1e-4, equal_nan=True)
    tiny = (again[odd[3]].double() - (x[odd[3]].double() @ w.double().t() + (0 if across else b.double()))).abs()
    assert (tiny <= bound[odd[3]] * 1e-34 + (0 if across else 2.0 ** -23 * b.double().abs())).all()
    same = torch.ones(N, dtype=torch.bool, device=dev)
    same[odd] = False
    assert ((again.double() - want).abs() <= bound)[same].all()


def test_product_with_the_weight_in_registers_and_more_odd_tiles_than_bits():
    """A workgroup remembers which of its tiles had odd sums in 256 bits; row 5 of the first tile and its namesake 256 tiles on share one."""
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    N = 32 * cus * 258 + 7
    x, wt = torch.randn(4096, 196, device=dev).repeat(N // 4096 + 1, 1)[:N].contiguous(), torch.randn(196, 132, device=dev)
    x[5, 7] = float("nan")
    got = projection._sum_of_products((x, wt))
    assert got[5].isnan().all() and got.isnan().sum() == 132
    first = 32 * cus * 256
    for rows in (slice(0, 5), slice(6, 64), slice(first, first + 64), slice(N - 64, N)):
        want = x[rows].double() @ wt.double()
        assert ((got[rows].double() - want).abs() <= 100 * 2.0 ** -23 * (x[rows].double().abs() @ wt.double().abs())).all()


@pytest.mark.parametrize("tiny,huge", [(-122, 100), (-140, 100), (-112, 33), (-109, 25)])
@pytest.mark.parametrize("across", [False, True])
def test_tiny_operands_with_large_partners_and_the_weight_in_registers(tiny, huge, across):
    """As test_tiny_operands_with_large_partners, with five tiles per workgroup: large weights in some columns of one wavefront; large rows in one tile
    each of five workgroups, the first, the second ... that it takes."""
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    N, K, O = 32 * cus * 5 - 7, 256, 250
    g = torch.Generator(device=dev).manual_seed(-tiny)
    product = lambda x, w: projection._sum_of_products((x, w.t().contiguous())) if across else projection._product(x, w, None)

    def close(got, want):
        return (got.double() - want).norm() <= 1e-6 * want.norm()                   # as for ordinary operands
    x, w = torch.randn(N, K, generator=g, device=dev) * 2.0 ** tiny, torch.randn(O, K, generator=g, device=dev)
    columns = torch.arange(40, 50, device=dev)
    w[columns] *= 2.0 ** huge
    assert close(product(x, w)[:, columns], x.double() @ w[columns].double().t())
    x, w = torch.randn(N, K, generator=g, device=dev), torch.randn(O, K, generator=g, device=dev) * 2.0 ** tiny
    large = torch.cat([32 * (i * cus + 3 * i + 1) + torch.arange(5, device=dev) for i in range(5)])
    x[large] *= 2.0 ** huge
    got, want = product(x, w)[large], x[large].double() @ w.double().t()
    for i in range(5):
        assert close(got[5 * i:5 * i + 5], want[5 * i:5 * i + 5]), i


@pytest.mark.parametrize("N,K,O", [(8192, 256, 256), (16500, 256, 512), (50001, 200, 250)])
@pytest.mark.parametrize("across", [False, True])
def test_kernels_agree_to_the_bit(N, K, O, across):
    """The same products and sums in the same order, whichever kernel a call's size takes: rows by themselves, in calls too small for the weight in registers."""
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(N + O)
    x, w, b = (torch.randn(*s, generator=g, device=dev) for s in ((N, K), (O, K), (O,)))
    wt = w.t().contiguous()
    product = lambda rows: projection._sum_of_products((rows, wt)) if across else projection._product(rows, w, b)
    got = product(x)
    for first in (0, 33, N - 4100):
        some = x[first:first + 4100].contiguous()
        assert torch.equal(product(some), got[first:first + 4100])


def _error(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("N,depth,width", [(4096, 64, 64), (5520, 256, 256), (16500, 512, 256), (4100, 1024, 1028), (8200, 2048, 516), (4096, 4096, 1024)])
@pytest.mark.parametrize("signs", ["random", "positive"])
def test_products_round_no_more_than_the_librarys(N, depth, width, signs):
    """Up to the deepest sums that the kernels take: the 2-norm error against float64 is no larger than the library's for the same product
    (measured: 0.63 to 0.87 of it from 256 terms on), and with random signs what the rounding of the sums alone makes.  Every other
    number of parts would show: two parts leave 2.3e-6 whatever the depth."""
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(depth)
    make = torch.randn if signs == "random" else torch.rand
    x, w = make(N, depth, generator=g, device=dev), make(width, depth, generator=g, device=dev)
    wt, want = w.t().contiguous(), x.double() @ w.double().t()
    for got, library in ((projection._product(x, w, None), torch.nn.functional.linear(x, w)), (projection._sum_of_products((x, wt)), x @ wt)):
        assert got is not None
        assert _error(got, want) <= 1.1 * _error(library, want)
        if signs == "random":
            # six roundings per 16 terms, each at most 2^-23 of a running sum of sqrt(terms so far) and 0.4 of that in size:
            # (6 / 16 depth)^(1/2) 0.4 2^-23 of the result, 3e-8 depth^(1/2)
            assert _error(got, want) <= 3e-8 * depth ** 0.5
    # the same terms dealt to several layers
    cut = depth // 4
    parts = tuple(t for i in range(4) for t in (x[:, i * cut:(i + 1) * cut].contiguous(), wt[i * cut:(i + 1) * cut].contiguous()))
    got = projection._sum_of_products(parts)
    if got is not None:
        assert _error(got, want) <= 1.1 * _error(x @ wt, want)
    assert got is not None or cut > 256


@pytest.mark.parametrize("N,widths", [(16500, (512, 256, 256)), (5520, (256, 64)), (33000, (512, 512, 512, 512))])
def test_gradient_of_rows_that_deep_layers_share(N, widths):
    """The offset and weight layers of the base model (512, 256 and 256 columns) and deeper sums, against the library's products and sums."""
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(N)
    gs = [torch.randn(N, o, generator=g, device=dev) for o in widths]
    ws = [torch.randn(o, 256, generator=g, device=dev) for o in widths]
    got = projection._sum_of_products(tuple(t for pair in zip(gs, ws) for t in pair))
    assert got is not None
    want = sum(a.double() @ b.double() for a, b in zip(gs, ws))
    assert _error(got, want) <= min(1.1 * _error(sum(a @ b for a, b in zip(gs, ws)), want), 3e-8 * sum(widths) ** 0.5)


@pytest.mark.parametrize("N", [4096, 184950, 600000])
@pytest.mark.parametrize("signs", ["random", "positive"])
def test_weight_gradients_round_no_more_than_the_librarys(N, signs):
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(N)
    make = torch.randn if signs == "random" else torch.rand
    x, y = make(N, 128, generator=g, device=dev), make(N, 64, generator=g, device=dev)
    got, bias = projection._weight_gradients(x, y, True)
    want = y.double().t() @ x.double()
    assert _error(got, want) <= 1.1 * _error(y.t().mm(x), want)
    assert _error(bias, y.double().sum(0)) <= 5e-7


@pytest.mark.parametrize("tiny,huge", [(-122, 100), (-140, 100), (-112, 33), (-120, 60), (-112, 31), (-109, 25)])
@pytest.mark.parametrize("mixed", [False, True])
def test_tiny_operands_with_large_partners(tiny, huge, mixed):
    """The lowest parts of the tiny operands are denormal numbers, or nothing is left of them at all; the sums are ordinary ones.  `mixed`:
    beside ordinary operands, in tiles of their own and in the same ones."""
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    torch.manual_seed(4)
    x, w, g = torch.randn(4200, 64, device=dev), torch.randn(96, 64, device=dev), torch.randn(4200, 96, device=dev)
    some = slice(100, 140) if mixed else slice(None)
    x[some] *= 2.0 ** tiny                                   # denormals of float32 are rounded here: the products are of what is left
    w *= 2.0 ** huge
    if mixed:
        x[:40, 5] *= 2.0 ** tiny
    rows = slice(some.start, some.stop) if mixed else slice(None)
    want = x.double() @ w.double().t()
    for got in (projection._product(x, w, None), projection._sum_of_products((x, w.t().contiguous())), projection._sum_of_products((x, w.t().contiguous()) * 2) / 2):
        # as ordinary operands (test_product): some 1e-7 of the 2-norm, each part of the rows by itself
        for part in (rows, slice(None)):
            assert (got[part].double() - want[part]).norm() <= 1e-6 * want[part].norm()
    g *= 2.0 ** huge
    got, _ = projection._weight_gradients(x, g, False)
    assert (got.double() - g.double().t() @ x.double()).norm() <= 1e-6 * (g.double().t() @ x.double()).norm()
    if mixed:
        g[:100], g[140:] = 0, 0                              # the tiny rows alone
        got, _ = projection._weight_gradients(x, g, False)
        assert (got.double() - g.double().t() @ x.double()).norm() <= 1e-6 * (g.double().t() @ x.double()).norm()


def test_gradients_that_are_no_numbers_take_no_walk():
    """A loss that is NaN or infinite leaves gradients of which every sum is formed again: by matrix instructions (measured: two or
    three times a finite step's time), not by one lane's loop over the rows per element (55 to 105 times)."""
    from dfa3D.modules import projection
    dev = torch.device("cuda:0")
    torch.manual_seed(2)
    x, w, b, g = (torch.randn(*s, device=dev) for s in ((20000, 256), (256, 256), (256,), (20000, 256)))
    bad = torch.full_like(g, float("nan"))

    def best(call):
        times = []
        for _ in range(5):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            call()
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)
    for call in (lambda t: projection._weight_gradients(x, t, True), lambda t: projection._sum_of_products((t, w)), lambda t: projection._product(t, w, b)):
        assert best(lambda: call(bad)) <= 12 * best(lambda: call(g))


@pytest.mark.parametrize("N,K,widths", [(4097, 64, (64,)), (5000, 36, (128, 66)), (4160, 256, (128, 64, 64)), (33001, 20, (4, 200, 72, 8))])
@pytest.mark.parametrize("train", [False, True])
def test_several_layers_on_the_same_rows(N, K, widths, train):
    from dfa3D.modules.projection import Projection, projections
    dev = torch.device("cuda:0")
    torch.manual_seed(N)
    layers = [Projection(K, O, library_forward=i == 1).to(dev) for i, O in enumerate(widths)]
    x = torch.randn(N, K, device=dev, requires_grad=train)
    gs = [torch.randn(N, O, device=dev) for O in widths]
    with torch.set_grad_enabled(train):
        got = projections(x, layers)
    xd = x.detach().double()
    for y, l in zip(got, layers):
        bound = (6 * (K // 16 + 1) + 18) * 2.0 ** -23 * (xd.abs() @ l.weight.detach().double().abs().t() + l.bias.detach().double().abs())
        assert ((y.detach().double() - (xd @ l.weight.detach().double().t() + l.bias.detach().double())).abs() <= bound).all()
    if not train:
        return
    params = [p for l in layers for p in (l.weight, l.bias)]
    grads = torch.autograd.grad(got, [x] + params, gs, retain_graph=True)
    want = sum(g.double() @ l.weight.detach().double() for g, l in zip(gs, layers))
    size = sum(g.double().abs() @ l.weight.detach().double().abs() for g, l in zip(gs, layers))
    # sums of at most 128 terms by the matrix unit, the rest to nearest (library products where a width is no multiple of four)
    assert ((grads[0].double() - want).abs() <= (6 * 9 + 18 + 2 * len(widths)) * 2.0 ** -23 * size).all()
    for i, (g, l) in enumerate(zip(gs, layers)):
        gw, gb = torch.autograd.grad(l(x), [l.weight, l.bias], g)
        assert torch.equal(grads[1 + 2 * i], gw) and torch.equal(grads[2 + 2 * i], gb)
    # one result's gradient alone; rows that want none; gradients of gradients
    gx, gw = torch.autograd.grad(got[-1], [x, layers[-1].weight], gs[-1], retain_graph=True)
    assert torch.equal(gw, grads[1 + 2 * (len(widths) - 1)])
    torch.testing.assert_close(gx.double(), gs[-1].double() @ layers[-1].weight.detach().double(), rtol=1e-4, atol=1e-4)
    gw, = torch.autograd.grad(projections(x.detach(), layers)[0], [layers[0].weight], gs[0])
    assert torch.equal(gw, grads[1])
    gw, = torch.autograd.grad(sum(y.square().sum() for y in got), [layers[0].weight], create_graph=True)
    assert torch.autograd.grad(gw.square().sum(), [x])[0].isfinite().all()


def test_layers_with_hooks_are_called():
    from dfa3D.modules.projection import Projection, projections
    dev = torch.device("cuda:0")
    layers = [Projection(64, 64).to(dev) for _ in range(2)]
    seen = []
    layers[1].register_forward_hook(lambda m, i, o: seen.append(o))
    x = torch.randn(5000, 64, device=dev)
    with torch.no_grad():
        got = projections(x, layers)
    assert len(seen) == 1 and seen[0] is got[1]


def test_offsets_keep_the_librarys_result():
    from dfa3D.modules.projection import Projection
    dev = torch.device("cuda:0")
    layer = Projection(256, 128, library_forward=True).to(dev)
    x = torch.randn(5000, 256, device=dev)
    want = torch.nn.functional.linear(x, layer.weight, layer.bias)
    assert torch.equal(layer(x), want)
    with torch.no_grad():
        assert torch.equal(layer(x), want)


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
    w, b = layer.weight.detach(), layer.bias.detach()
    x = x.detach()
    from dfa3D.modules.projection import _product
    assert _product(x, w, b) is not None
    for args in ((x, layer.weight, b), (x.double(), w, b), (x.t(), w, b), (x, w, b[:-1]), (x[:, :-2].contiguous(), w, b), (x[0], w, b),
                 (x, w[:-1].contiguous(), None), (x, w.t(), None), (torch._neg_view(x), w, b), (x[:0], w, b)):
        assert _product(*args) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert _product(x, w, b) is None
    few = torch.randn(7, 64, device=dev)
    torch.autograd.grad(layer(few).sum(), [layer.weight])
