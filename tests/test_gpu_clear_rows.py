"""The blocks beside the bin scan that clear what the tile kernel only adds to: rows of a batch element that are no multiple of a
wavefront's 64 (or 16, below 2^18 rows), rows in pieces of 4 and of 16 bytes, heads that do not divide 64, maps of one pixel row or column."""
import pytest
import torch

from test_gpu_parity import _dev, tiny_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,C,D,levels", [
    (1, 4, 3, ((1, 1),)), (3, 5, 7, ((1, 67), (29, 1))), (6, 20, 59, ((37, 67), (19, 34), (10, 17))),
    (5, 12, 9, ((3, 5),)), (8, 64, 16, ((13, 19), (2, 2))),
    (8, 8, 4, ((128, 127),)), (8, 8, 5, ((128, 128), (1, 1))), (7, 4, 4, ((200, 190),)),      # 260096, 262160 and 266000 rows with B = 2, 2 and 1
], ids=str)
def test_buffers_that_held_nan(M, C, D, levels):
    from dfa3D import _ext
    dev = _dev()
    B = 1 if M == 7 else 2
    t = tiny_case(77, B=B, M=M, C=C, D=D, Q=300, P=3, levels=levels, dtype=torch.float32)
    t["loc"][..., 0] *= 0.4                              # some tiles stay without points
    value, dist, loc, attn, go, shapes, lsi = [t[k].to(dev) for k in ("value", "dist", "loc", "attn", "grad_out", "shapes3", "lsi")]

    def run(fill, clear):
        gv, gd = torch.full_like(value, fill), torch.full_like(dist, fill)
        _ext.dfa3d_fused_backward(value, dist, shapes, lsi, loc, attn, go, None, gv, gd, torch.empty_like(loc), torch.empty_like(attn), 64,
                                  clear=clear)
        return gv.cpu(), gd.cpu()

    for got, want in zip(run(float("nan"), True), run(0.0, False)):
        assert torch.equal(got == 0, want == 0)          # NaN nowhere, and nothing cleared that was written
        # up to 300 * 3 terms in another order: 900 roundings of 2^-24 of the largest sum
        assert (got - want).abs().max() <= 900 * 2 ** -24 * want.abs().max()
