"""Counting and filling the bins: blocks that take one turn of 2048 points, several, or none; turns that end inside a unit's
points; units of exactly a turn; and one point more than that, which the sorted form does not take."""
import pytest
import torch

from test_gpu_parity import _dev, tiny_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,M,Q,P,levels", [
    (1, 1, 1, 1, ((4, 5),)), (3, 5, 2049, 1, ((9, 14),)), (1, 6, 2731, 3, ((9, 14), (3, 2))),
    (2, 8, 5000, 16, ((21, 30),)),                       # 640 turns: more than the chip holds blocks
    (5, 3, 4800, 15, ((21, 30),)),                       # 540 turns, the last of each batch element and head not full
    (1, 3, 300, 2048, ((21, 30),)), (1, 2, 40, 2049, ((21, 30),)),
], ids=str)
def test_every_point_is_visited_once(B, M, Q, P, levels):
    from dfa3D import _ext
    dev = _dev()
    t = tiny_case(91, B=B, M=M, C=4, D=4, Q=Q, P=P, levels=levels, dtype=torch.float32)
    t = {k: v.to(dev) for k, v in t.items() if torch.is_tensor(v)}
    t["grad_out"] = t["grad_out"].abs() + 0.5            # sums without cancellation

    def run(dtype):
        v, d, loc, attn, go = (t[k].to(dtype) for k in ("value", "dist", "loc", "attn", "grad_out"))
        loc, attn = t["loc"].to(dtype), t["attn"].to(dtype)
        gl, ga = torch.full_like(loc, float("nan")), torch.full_like(attn, float("nan"))
        gv, gd = torch.zeros_like(v), torch.zeros_like(d)
        _ext.dfa3d_fused_backward(v, d, t["shapes3"], t["lsi"], loc, attn, go, None, gv, gd, gl, ga, 64)
        return [x.double().cpu() for x in (gv, gd, gl, ga)]

    got, want = run(torch.float32), run(torch.float64)
    # per point: a few dozen operations on numbers of the size of the largest result
    for x, y in zip(got[2:], want[2:]):
        assert (x - y).abs().max() <= 256 * 2 ** -24 * y.abs().max()
    # per pixel: up to the points of a batch element, head and level in any order, rounded once each
    for x, y in zip(got[:2], want[:2]):
        assert (x - y).abs().max() <= max(64, Q * P) * 2 ** -24 * y.abs().max()
        assert abs(x.sum() - y.sum()) <= 1e-5 * y.abs().sum()
