"""Products and sums with few rows, whose sums are split over wavefronts: rows, columns and depths around its tiles and steps, both ways the weight may lie,
several layers of unlike depths, operands that are no ordinary numbers, and both sides of the line to the kernels of larger tiles."""
import pytest
import torch

from dfa3D import _lib

pytestmark = pytest.mark.gpu


def _rand(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _product(x, w, b=None, addend=None):
    y, p = torch.full((len(x), len(w)), float("nan"), device="cuda"), _lib.ptr
    rc = _lib.lib().dfa3d_linear_add(p(x), p(w), p(b), p(addend), p(y), len(x), len(w), x.shape[1], _lib.stream_of(x))
    _lib.check(rc, "dfa3d_linear_add")
    return y


def _sum(pairs):
    g, w = pairs[0]
    y = torch.full((len(g), w.shape[1]), float("nan"), device="cuda")
    sets = (_lib.LinearSet * len(pairs))(*((_lib.ptr(w), _lib.ptr(g), g.shape[1]) for g, w in pairs))
    _lib.check(_lib.lib().dfa3d_linear_sum(sets, len(pairs), _lib.ptr(y), len(g), w.shape[1], _lib.stream_of(g)), "dfa3d_linear_sum")
    return y


def _within_roundings(got, terms, more=()):
    """terms: pairs of factors.  n products and their sum: a rounding of 2^-24 of the sum of the sizes each."""
    want = sum(a.double() @ b.double() for a, b in terms) + sum(m.double() for m in more)
    size = sum(a.double().abs() @ b.double().abs() for a, b in terms) + sum(m.double().abs() for m in more)
    n = sum(a.shape[1] for a, _ in terms) + len(more)
    assert ((got - want).abs() <= n * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("N", [1, 31, 32, 33, 65, 300])
@pytest.mark.parametrize("cols,depth", [(2, 128), (30, 132), (34, 252), (258, 260), (64, 1028), (128, 4096)])
def test_product(N, cols, depth):
    g = torch.Generator(device="cuda").manual_seed(N + cols + depth)
    x, w, b, r = _rand(g, N, depth), _rand(g, cols, depth), _rand(g, cols), _rand(g, N, cols)
    _within_roundings(_product(x, w), [(x, w.t())])
    _within_roundings(_product(x, w, b, r), [(x, w.t())], (b.expand(N, -1), r))
    assert torch.equal(_product(x, w, b, r), _product(x, w, b) + r) and torch.equal(_product(x, w, b), _product(x, w, b))


@pytest.mark.parametrize("N", [1, 33, 300])
@pytest.mark.parametrize("cols,widths", [(2, (4,)), (36, (4, 12, 60, 68)), (64, (260,)), (256, (512, 256, 256)), (130, (1024, 4)), (34, (64, 64, 64, 16))])
def test_sums(N, cols, widths):
    g = torch.Generator(device="cuda").manual_seed(N + cols)
    pairs = [(_rand(g, N, d), _rand(g, d, cols)) for d in widths]
    got = _sum(pairs)
    _within_roundings(got, pairs)
    assert torch.equal(got, _sum(pairs))


@pytest.mark.parametrize("across", [False, True])
def test_operands_that_are_no_ordinary_numbers(across):
    """As float32 arithmetic has it: infinities and NaN where they meet, the largest numbers, tiny ones with large partners."""
    g = torch.Generator(device="cuda").manual_seed(3)
    x, w = _rand(g, 70, 256), _rand(g, 256, 40)
    x[3, 5], x[10, 200], x[40, 17], w[9, 33] = float("inf"), float("nan"), 3.4e38, float("-inf")
    x[64] *= 2.0 ** -120
    x[65], w[:, 7] = 2.0 ** -140, 2.0 ** 100
    got = _sum([(x, w)]) if across else _product(x, w.t().contiguous())
    want = x.double() @ w.double()
    clear = torch.isfinite(want) & (want.abs() < 3e38)
    clear[40], clear[:, 33] = False, False                    # next to overflow, and infinite
    clear[65] &= want[65].abs() >= 2.0 ** -89                 # smaller sums of denormal operands may lose them (include/dfa3d.h)
    assert torch.equal(torch.isnan(got[:, 33]), torch.isnan(want[:, 33])) and torch.isnan(got[10]).all()
    assert torch.equal(got[3].isinf(), want[3].isinf()) and torch.equal(got[3].sign(), want[3].float().sign())
    finite = x.double().nan_to_num(0, 0, 0).abs() @ w.double().nan_to_num(0, 0, 0).abs()
    assert ((got - want).abs() <= 256 * 2.0 ** -24 * finite + 2.0 ** -149)[clear].all()


@pytest.mark.parametrize("N,cols,depth,across", [(1536, 256, 256, False), (1537, 256, 256, False), (8192, 256, 512, True), (4096, 256, 512, True), (4097, 256, 512, True)])
def test_both_sides_of_the_line(N, cols, depth, across):
    """The two kernels' sums are the same products in another order."""
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w = _rand(g, N, depth), _rand(g, depth, cols)
    part = slice(N - 200, N)
    if across:
        got, few = _sum([(x, w)])[part], _sum([(x[part].contiguous(), w)])
    else:
        w = w.t().contiguous()
        got, few = _product(x, w)[part], _product(x[part].contiguous(), w)
        w = w.t()
    for y in (got, few):
        _within_roundings(y, [(x[part], w)])


def test_replayed_in_a_graph():
    g = torch.Generator(device="cuda").manual_seed(1)
    x, w, b, r = _rand(g, 100, 256), _rand(g, 64, 256), _rand(g, 64), _rand(g, 100, 64)
    pairs = [(_rand(g, 100, d), _rand(g, d, 64)) for d in (128, 68)]
    call = lambda: (_product(x, w, b, r), _sum(pairs))
    call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for _ in range(3):
        x.copy_(_rand(g, 100, 256))
        pairs[0][0].copy_(_rand(g, 100, 128))
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, e) for a, e in zip(out, call()))
