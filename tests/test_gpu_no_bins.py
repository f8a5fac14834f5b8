"""Level tables the binning has no bins for: many levels on one map (more tiles than the counters hold), and a table none of
whose levels fits the keys.  The tile kernels then add point by point, and every gradient is written all the same."""
import pytest
import torch

from forms import tiny_case
from test_gpu_parity import (F32_BWD, F32_FWD, _as_inputs, _assert_sums_within_term_count_bound, _dev, _gpu_one_stage,
                             _gpu_two_stage, _oracle_one_stage)

pytestmark = pytest.mark.gpu


def _one_map_for_all_levels(C, D, P=3):
    """14 levels of 16 x 16 on the same 256 keys: 14 x 9 tiles of 8 x 8 (more of smaller ones) where the counters hold 65."""
    inp = _as_inputs(tiny_case(seed=90 + C, B=2, M=3, C=C, D=D, Q=40, P=P, levels=((16, 16),) * 14, dtype=torch.float32))
    inp["level_start_index"].zero_()
    inp["value"], inp["value_dpt_dist"] = inp["value"][:, :256].contiguous(), inp["value_dpt_dist"][:, :256].contiguous()
    return inp


@pytest.mark.parametrize("C,D,P", [(32, 64, 3), (20, 41, 3), (96, 16, 3), (8, 4, 150)],
                         ids=["cells", "odd-bins", "row-owned", "2100-points-per-unit"])
def test_more_tiles_than_counters(oracle, C, D, P):
    dev = _dev()
    inp = _one_map_for_all_levels(C, D, P)
    want = _oracle_one_stage(oracle, inp)
    for got in (_gpu_one_stage(inp, dev), _gpu_two_stage(inp, dev, sliced=False)):
        for i in (0, 1, 4, 5):
            torch.testing.assert_close(got[i], want[i], **(F32_FWD if i < 2 else F32_BWD))
        _assert_sums_within_term_count_bound(oracle, inp, got[2], got[3])


def test_gradients_arriving_at_every_output(oracle):
    """A shared distribution with the weight_update output, and the depth scores' own gradient."""
    from test_gpu_parity import _shared_dist_expectation
    from dfa3D.functional import MultiScale3DDeformableAttnWeightUpdateFunction
    dev = _dev()
    inp = _one_map_for_all_levels(32, 16)
    go_score = torch.randn(2, 40, 3, 14, 3, 4, generator=torch.Generator().manual_seed(4))
    args = [inp[k] for k in ("value", "value_dpt_dist", "spatial_shapes", "level_start_index", "sampling_locations", "attention_weights")]
    want = _oracle_one_stage(oracle, inp)
    gd_score, gl_score = oracle.depth_score_backward(inp["value_dpt_dist"], inp["spatial_shapes"], inp["level_start_index"],
                                                     inp["sampling_locations"], go_score)
    got = _gpu_one_stage(inp, dev, grad_score=go_score)
    torch.testing.assert_close(got[3], want[3] + gd_score, **F32_BWD)
    torch.testing.assert_close(got[4], want[4] + gl_score, **F32_BWD)
    inp["value_dpt_dist"] = inp["value_dpt_dist"][:, :, :1].contiguous()
    grad_wu = torch.randn(2, 40, 3, 1, generator=torch.Generator().manual_seed(5))
    want = _shared_dist_expectation(oracle, inp, grad_wu=grad_wu)
    leaves = [inp[k].to(dev).requires_grad_() for k in ("value", "value_dpt_dist", "sampling_locations", "attention_weights")]
    out, wu = MultiScale3DDeformableAttnWeightUpdateFunction.apply(leaves[0], leaves[1], args[2].to(dev), args[3].to(dev),
                                                                   leaves[2], leaves[3], 64)
    grads = torch.autograd.grad([out, wu], leaves, [inp["grad_output"].to(dev), grad_wu.to(dev)])
    for g, w in zip(grads, want[3:]):
        torch.testing.assert_close(g.cpu(), w, **F32_BWD)


def test_bfloat16_gradients(oracle):
    dev = _dev()
    from dfa3D import _ext
    inp = _one_map_for_all_levels(32, 64)
    r16 = dict(inp, **{k: inp[k].bfloat16().float() for k in ("value", "value_dpt_dist", "grad_output")})
    v, d, go = (r16[k].bfloat16().to(dev) for k in ("value", "value_dpt_dist", "grad_output"))
    loc, attn = inp["sampling_locations"].to(dev), inp["attention_weights"].to(dev)
    nan = lambda like: torch.full_like(like, float("nan"))
    gv, gd, gl, ga = nan(v), nan(d), nan(loc), nan(attn)
    _ext.dfa3d_fused_backward(v, d, inp["spatial_shapes"].to(dev), inp["level_start_index"].to(dev), loc, attn, go, None, gv, gd,
                              gl, ga, 64, clear=True)
    want = _oracle_one_stage(oracle, r16)
    torch.testing.assert_close(gl.cpu(), want[4], **F32_BWD)
    torch.testing.assert_close(ga.cpu(), want[5], **F32_BWD)
    # every add rounds the stored sum: the bound is (number of terms) * 2^-9 of the terms' sum, which the rms stays far inside
    for g, w in ((gv, want[2]), (gd, want[3])):
        rel = ((g.float().cpu() - w).pow(2).sum() / w.pow(2).sum()).sqrt().item()
        assert rel < 0.1, rel


@pytest.mark.parametrize("C", [32, 96])
def test_no_usable_level(C):
    """Every point is skipped: zero gradients, whatever the buffers held."""
    dev = _dev()
    from dfa3D import _ext
    t = tiny_case(seed=93, B=1, M=2, C=C, D=8, Q=30, P=4, levels=((6, 5),), dtype=torch.float32)
    shapes = torch.tensor([[6, 50, 8]], device=dev)                      # 300 keys where there are 30
    v, d, loc, attn, go = (t[k].to(dev) for k in ("value", "dist", "loc", "attn", "grad_out"))
    lsi = t["lsi"].to(dev)
    nan = lambda like: torch.full_like(like, float("nan"))
    gv, gd, gl, ga = nan(v), nan(d), nan(loc), nan(attn)
    _ext.dfa3d_fused_backward(v, d, shapes, lsi, loc, attn, go, None, gv, gd, gl, ga, 64, clear=True)
    for g in (gv, gd, gl, ga):
        assert (g == 0).all()
    gv, gl, ga, gs = nan(v), nan(loc)[..., :2].contiguous(), nan(attn), torch.full((*attn.shape, 4), float("nan"), device=dev)
    _ext.wms_deform_attn_backward_into(v, shapes[:, :2].contiguous(), lsi, loc[..., :2].contiguous(), attn, torch.ones_like(gs), go,
                                       gv, gl, ga, gs, im2col_step=64, clear=True)
    for g in (gv, gl, ga, gs):
        assert (g == 0).all()
    gd, gl = nan(d), nan(loc)
    _ext.ms_depth_score_sample_backward_into(d, shapes, lsi, loc, torch.ones_like(gs), gd, gl, 64, clear=True)
    assert (gd == 0).all() and (gl == 0).all()
