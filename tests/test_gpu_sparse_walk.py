"""Tile kernel, bfloat16 storage: below three quarters of a point per pixel the walkers take one point of a pixel at a time, else four
(lists of 0 to 3 points and a long one on both sides of that line, pixels with one point or none on a large map, rows that are not finite)."""
import pytest
import torch

from test_gpu_parity import _assert_per_point_within_term_count_bound, _assert_sums_within_term_count_bound, _dev

pytestmark = pytest.mark.gpu


def _inputs(C, D, H, W, count, M=2, seed=0):
    """One level; pixel i is the upper left one of count[i] points."""
    g = torch.Generator().manual_seed(seed + C)
    pixel = torch.repeat_interleave(torch.arange(H * W), count)
    pixel = pixel[torch.randperm(len(pixel), generator=g)]
    frac = torch.rand(len(pixel), 2, generator=g) * 0.8 + 0.1
    x, y = ((pixel % W) + 0.5 + frac[:, 0]) / W, ((pixel // W) + 0.5 + frac[:, 1]) / H
    loc = torch.stack([x, y, torch.rand(len(pixel), generator=g)], -1).view(1, -1, 1, 1, 1, 3).repeat(1, 1, M, 1, 1, 1)
    Q = loc.shape[1]
    r16 = lambda *s: torch.randn(*s, generator=g).bfloat16().float()
    return {"value": r16(1, H * W, M, C), "value_dpt_dist": torch.rand(1, H * W, M, D, generator=g).bfloat16().float(),
            "spatial_shapes": torch.tensor([[H, W, D]]), "level_start_index": torch.tensor([0]), "sampling_locations": loc,
            "attention_weights": torch.rand(1, Q, M, 1, 1, generator=g), "grad_output": r16(1, Q, M * C)}


def _forward_of(oracle, inp):
    return oracle.dfa3d_forward(*(inp[k] for k in ("value", "value_dpt_dist", "spatial_shapes", "level_start_index",
                                                    "sampling_locations", "attention_weights")))


def _fused(inp, dev):
    from dfa3D import _ext
    t = {k: v.to(dev) for k, v in inp.items()}
    value, dist, go = (t[k].bfloat16() for k in ("value", "value_dpt_dist", "grad_output"))
    gv, gd = torch.zeros(value.shape, device=dev), torch.zeros(dist.shape, device=dev)
    gl, ga = torch.empty_like(t["sampling_locations"]), torch.empty_like(t["attention_weights"])
    _ext.dfa3d_fused_backward(value, dist, t["spatial_shapes"], t["level_start_index"], t["sampling_locations"], t["attention_weights"],
                              go, None, gv, gd, gl, ga, 64)
    return gv.cpu(), gd.cpu(), gl.cpu(), ga.cpu()


@pytest.mark.parametrize("short", [0, 1])
@pytest.mark.parametrize("C", [8, 20, 24, 32, 36, 48, 64])
def test_both_sides_of_the_line(oracle, C, short):
    """16 x 24 pixels with 288 points (three quarters each: four at a time) and 287, in lists of 0 to 3 and one of 40."""
    H, W = 16, 24
    count = torch.zeros(H * W, dtype=torch.long)
    count[5::8] = 2
    count[2::13] = 3
    count[W + 7] = 40
    rest = 288 - short - int(count.sum())
    assert rest > 0
    count[(count == 0).nonzero()[:rest, 0]] = 1
    inp = _inputs(C, 16, H, W, count)
    assert inp["grad_output"].shape[1] == 288 - short
    gv, gd, gl, ga = _fused(inp, _dev())
    out, score = _forward_of(oracle, inp)
    _assert_per_point_within_term_count_bound(oracle, inp, out, score, gl, ga)
    _assert_sums_within_term_count_bound(oracle, inp, gv, gd)


@pytest.mark.parametrize("every", [2, 7])
@pytest.mark.parametrize("C,D", [(16, 8), (20, 9), (32, 16), (64, 8)])
def test_one_point_per_pixel_on_a_large_map(oracle, C, D, every):
    H, W = 97, 131
    count = (torch.arange(H * W) % every == 0).long()
    inp = _inputs(C, D, H, W, count, M=1)
    gv, gd, gl, ga = _fused(inp, _dev())
    out, score = _forward_of(oracle, inp)
    _assert_per_point_within_term_count_bound(oracle, inp, out, score, gl, ga)
    _assert_sums_within_term_count_bound(oracle, inp, gv, gd)


@pytest.mark.parametrize("C", [24, 32, 64])
def test_stage_two_alone_on_a_sparse_map(oracle, C):
    """Without depth tile: equal scores of one make the fused operator's distribution a single bin of ones."""
    from dfa3D import _ext
    H, W, M, dev = 61, 83, 2, _dev()
    inp = _inputs(C, 1, H, W, (torch.arange(H * W) % 3 == 0).long(), M=M)
    inp["value_dpt_dist"] = torch.ones_like(inp["value_dpt_dist"])
    inp["sampling_locations"][..., 2] = 0.5                  # the centre of the only bin: every score is one
    t = {k: v.to(dev) for k, v in inp.items()}
    loc2 = t["sampling_locations"][..., :2].contiguous()
    gv = torch.zeros(inp["value"].shape, device=dev)
    gl, ga = torch.empty_like(loc2), torch.empty_like(t["attention_weights"])
    _ext.ms_deform_attn_backward(t["value"].bfloat16(), t["spatial_shapes"][:, :2].contiguous(), t["level_start_index"], loc2,
                                 t["attention_weights"], t["grad_output"].bfloat16(), gv, gl, ga, 64)
    out, score = _forward_of(oracle, inp)
    whole = torch.zeros(inp["sampling_locations"].shape)
    whole[..., :2] = gl.cpu()
    want = oracle.dfa3d_backward(*(inp[k] for k in ("value", "value_dpt_dist", "spatial_shapes", "level_start_index",
                                                     "sampling_locations", "attention_weights")), score, inp["grad_output"])
    whole[..., 2] = want[2][..., 2]                          # no depth here
    _assert_per_point_within_term_count_bound(oracle, inp, out, score, whole, ga.cpu())
    _assert_sums_within_term_count_bound(oracle, inp, gv.cpu(), want[1])


@pytest.mark.parametrize("C", [32, 64])
def test_rows_that_are_not_finite_stay_with_their_pixels(C):
    """Infinities and NaN in a few queries' gradients reach the pixels and points of those queries and no others."""
    H, W, dev = 45, 67, _dev()
    inp = _inputs(C, 8, H, W, (torch.arange(H * W) % 5 == 0).long() * 2)
    plain = _fused(inp, dev)
    M, Q = 2, inp["grad_output"].shape[1]
    go = inp["grad_output"].clone().view(1, Q, M, C)
    hit = torch.tensor([3, Q // 2, Q - 1])
    go[0, hit, :, 1] = torch.tensor([float("inf"), float("nan"), float("-inf")])[:, None]
    gv, gd, gl, ga = _fused(dict(inp, grad_output=go.view(1, Q, M * C)), dev)
    loc = inp["sampling_locations"][0, :, 0, 0, 0]
    x0, y0 = (loc[:, 0] * W - 0.5).floor().long(), (loc[:, 1] * H - 0.5).floor().long()
    touched = torch.zeros(H * W, dtype=torch.bool)
    for q in hit.tolist():
        for dy in (0, 1):
            for dx in (0, 1):
                if y0[q] + dy < H and x0[q] + dx < W:
                    touched[(y0[q] + dy) * W + x0[q] + dx] = True
    others = torch.ones(Q, dtype=torch.bool)
    others[hit] = False
    assert not torch.isfinite(gv[0, touched][..., 1]).any()      # every weight is positive
    assert torch.isfinite(gv[0][..., [c for c in range(C) if c != 1]]).all()
    for a, b in ((gv[0, ~touched], plain[0][0, ~touched]), (gl[0, others], plain[2][0, others]), (ga[0, others], plain[3][0, others])):
        assert torch.isfinite(a).all()
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)      # sums in another order
    assert torch.isfinite(gd[0, ~touched]).all() and not torch.isfinite(ga[0, hit]).any()
