"""Tile kernel, bfloat16 storage: its walkers take the points of a pixel four at a time.  Pixels with 0 to 9 points each, on every
lane grouping and on rows shorter than their lane group, and rows that are not finite."""
import pytest
import torch

from test_gpu_parity import _assert_per_point_within_term_count_bound, _assert_sums_within_term_count_bound, _dev

pytestmark = pytest.mark.gpu


def _inputs(C, D, H=13, W=19, M=2, seed=0):
    """One level; pixel i is the upper left one of i % 10 points."""
    g = torch.Generator().manual_seed(seed + C)
    pixel = torch.repeat_interleave(torch.arange(H * W), torch.arange(H * W) % 10)
    pixel = pixel[torch.randperm(len(pixel), generator=g)]
    frac = torch.rand(len(pixel), 2, generator=g) * 0.8 + 0.1
    x, y = ((pixel % W) + 0.5 + frac[:, 0]) / W, ((pixel // W) + 0.5 + frac[:, 1]) / H
    loc = torch.stack([x, y, torch.rand(len(pixel), generator=g)], -1).view(1, -1, 1, 1, 1, 3).repeat(1, 1, M, 1, 1, 1)
    Q = loc.shape[1]
    r16 = lambda *s: torch.randn(*s, generator=g).bfloat16().float()
    return {"value": r16(1, H * W, M, C), "value_dpt_dist": torch.rand(1, H * W, M, D, generator=g).bfloat16().float(),
            "spatial_shapes": torch.tensor([[H, W, D]]), "level_start_index": torch.tensor([0]), "sampling_locations": loc,
            "attention_weights": torch.rand(1, Q, M, 1, 1, generator=g), "grad_output": r16(1, Q, M * C)}


def _backward(inp, dev):
    from dfa3D import _ext
    t = {k: v.to(dev) for k, v in inp.items()}
    value, dist, go = (t[k].bfloat16() for k in ("value", "value_dpt_dist", "grad_output"))
    gv, gd = torch.zeros(value.shape, device=dev), torch.zeros(dist.shape, device=dev)
    gl, ga = torch.empty_like(t["sampling_locations"]), torch.empty_like(t["attention_weights"])
    _ext.dfa3d_fused_backward(value, dist, t["spatial_shapes"], t["level_start_index"], t["sampling_locations"], t["attention_weights"],
                              go, None, gv, gd, gl, ga, 64)
    return gv.cpu(), gd.cpu(), gl.cpu(), ga.cpu()


@pytest.mark.parametrize("C,D", [(4, 3), (12, 16), (16, 64), (20, 8), (32, 64), (36, 16), (64, 9)])
def test_pixels_with_zero_to_nine_points(oracle, C, D):
    inp = _inputs(C, D)
    gv, gd, gl, ga = _backward(inp, _dev())
    out, score = oracle.dfa3d_forward(*(inp[k] for k in ("value", "value_dpt_dist", "spatial_shapes", "level_start_index",
                                                          "sampling_locations", "attention_weights")))
    _assert_per_point_within_term_count_bound(oracle, inp, out, score, gl, ga)
    _assert_sums_within_term_count_bound(oracle, inp, gv, gd)


@pytest.mark.parametrize("C", [16, 32, 64])
def test_rows_that_are_not_finite_stay_with_their_pixels(C):
    """Infinities and NaN in a few queries' gradients reach the pixels and points of those queries and no others."""
    inp = _inputs(C, 8)
    dev = _dev()
    plain = _backward(inp, dev)
    M, Q = 2, inp["grad_output"].shape[1]
    go = inp["grad_output"].clone().view(1, Q, M, C)
    hit = torch.tensor([3, Q // 2, Q - 1])
    go[0, hit, :, 1] = torch.tensor([float("inf"), float("nan"), float("-inf")])[:, None]
    gv, gd, gl, ga = _backward(dict(inp, grad_output=go.view(1, Q, M * C)), dev)
    H, W = inp["spatial_shapes"][0, :2].tolist()
    loc = inp["sampling_locations"][0, :, 0, 0, 0]
    x0, y0 = (loc[:, 0] * W - 0.5).floor().long(), (loc[:, 1] * H - 0.5).floor().long()
    touched = torch.zeros(H * W, dtype=torch.bool)
    for q in hit.tolist():
        for dy in (0, 1):
            for dx in (0, 1):
                if 0 <= y0[q] + dy < H and 0 <= x0[q] + dx < W:
                    touched[(y0[q] + dy) * W + x0[q] + dx] = True
    others = torch.ones(Q, dtype=torch.bool)
    others[hit] = False
    assert not torch.isfinite(gv[0, touched][..., 1]).any()      # every weight is positive
    assert torch.isfinite(gv[0][..., [c for c in range(C) if c != 1]]).all()
    for a, b in ((gv[0, ~touched], plain[0][0, ~touched]), (gl[0, others], plain[2][0, others]), (ga[0, others], plain[3][0, others])):
        assert torch.isfinite(a).all()
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)      # sums in another order
    assert torch.isfinite(gd[0, ~touched]).all() and not torch.isfinite(ga[0, hit]).any()
