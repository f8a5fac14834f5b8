"""Entry points of the C interface, or forms of their arguments, that the package itself has no use for."""
import pytest
import torch

from dfa3D import _lib

pytestmark = pytest.mark.gpu


def _stream():
    return torch.cuda.current_stream().cuda_stream


def test_lists_without_totals():
    g = torch.Generator().manual_seed(0)
    hit = (torch.rand(3, 2500, generator=g) < 0.3).cuda()
    longest, p = int(hit.sum(1).max()), _lib.ptr
    got = []
    for totals in (None, torch.full((3,), -7, dtype=torch.int32, device="cuda")):
        index, pos = (torch.full((3, n), 99, dtype=torch.int32, device="cuda") for n in (longest, 2500))
        _lib.check(_lib.lib().dfa3d_camera_index(p(hit), p(totals), p(index), p(pos), 3, 2500, longest, _stream()), "dfa3d_camera_index")
        got.append((index, pos))
    for index, pos in got:
        for cam in range(3):
            seen = hit[cam].nonzero()[:, 0].int()
            assert torch.equal(index[cam, :len(seen)], seen) and (index[cam, len(seen):] == -1).all()
            assert torch.equal(pos[cam][hit[cam]], torch.arange(len(seen), dtype=torch.int32, device="cuda")) and (pos[cam][~hit[cam]] == -1).all()


@pytest.mark.parametrize("N,O,K", [(1, 2, 4), (65, 130, 100), (9000, 256, 256)])
@pytest.mark.parametrize("bias", [True, False])
def test_linear_is_linear_add_without_addend(N, O, K, bias):
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w, b = (torch.randn(*s, generator=g, device="cuda") for s in ((N, K), (O, K), (O,)))
    p, b = _lib.ptr, b if bias else None
    y, y_add = (torch.full((N, O), float("nan"), device="cuda") for _ in range(2))
    _lib.check(_lib.lib().dfa3d_linear(p(x), p(w), p(b), p(y), N, O, K, _stream()), "dfa3d_linear")
    _lib.check(_lib.lib().dfa3d_linear_add(p(x), p(w), p(b), None, p(y_add), N, O, K, _stream()), "dfa3d_linear_add")
    assert torch.equal(y, y_add)
    want = x.double() @ w.double().t() + (b.double() if bias else 0)
    # K products and their sum: K roundings of 2^-24 of the sum of the sizes, and the bias
    size = x.double().abs() @ w.double().abs().t() + (b.double().abs() if bias else 0)
    assert ((y - want).abs() <= (K + 1) * 2.0 ** -24 * size).all()
    assert _lib.lib().dfa3d_linear(p(x), p(w), p(b), p(y), N, O, K + 2, _stream()) == -1        # no whole groups of four
