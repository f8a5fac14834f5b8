"""Forward with the value rows of a (batch, head) in LDS (small maps with many points): row lengths on both sides of every lane
group, points per unit from one to more than a wavefront holds, a last share of the queries that is not full, and maps on both sides
of what LDS holds.  Walking several groups per wavefront on request (iters = 2) keeps the gathers from memory, which form the same sums
in the same order."""
import pytest
import torch

from forms import tiny_case
from test_gpu_parity import F32_FWD, _as_inputs, _dev

pytestmark = pytest.mark.gpu


def _on(dev, t, store):
    return (t["value"].to(store).to(dev), t["value_dpt_dist"].to(store).to(dev), t["spatial_shapes"].to(dev), t["level_start_index"].to(dev),
            t["sampling_locations"].float().to(dev), t["attention_weights"].float().to(dev))


@pytest.mark.parametrize("L,P,C,Q", [(1, 1, 32, 2111), (1, 3, 4, 1501), (2, 4, 20, 611), (2, 5, 12, 397), (1, 8, 64, 640), (2, 4, 36, 513), (2, 16, 32, 129),
                                     (2, 33, 16, 70), (1, 10, 8, 777)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_against_the_oracle(oracle, L, P, C, Q, dtype):
    from dfa3D import _ext
    t = _as_inputs(tiny_case(seed=31 * C + P, B=2, M=3, C=C, D=7, Q=Q, P=P, levels=((5, 7), (3, 3))[:L]))
    value, dist, sh, lsi, loc, attn = _on(_dev(), t, dtype)
    got, score, wu = _ext.dfa3d_fused_forward(value, dist, sh, lsi, loc, attn, 64, need_depth_score=True, need_weight_update=True)
    cpu = [x.cpu() for x in (value, dist, sh, lsi, loc, attn)]
    want, want_score = oracle.dfa3d_forward(cpu[0].float(), cpu[1].float(), *cpu[2:])
    tol = F32_FWD if dtype == torch.float32 else dict(rtol=2 ** -8, atol=1e-5)         # stored in bfloat16: one rounding
    torch.testing.assert_close(got.cpu().float(), want, **tol)
    torch.testing.assert_close(score.cpu().float(), want_score, **tol)
    want_wu = (want_score.mean(-1) * cpu[5]).flatten(-2).sum(-1, keepdim=True)
    torch.testing.assert_close(wu.cpu().view_as(want_wu), want_wu, **{**tol, **F32_FWD})
    from dfa3D import _lib
    with _lib.launch_options(iters=2):
        again = _ext.dfa3d_fused_forward(value, dist, sh, lsi, loc, attn, 64, need_depth_score=True, need_weight_update=True)
    for a, b in zip((got, score, wu), again):
        assert torch.equal(a, b)


@pytest.mark.parametrize("levels,C,dtype", [(((21, 47),), 32, torch.float32), (((26, 38),), 32, torch.float32), (((19, 26),), 64, torch.float32),
                                            (((40, 49), (4, 3)), 32, torch.bfloat16), (((30, 41),), 24, torch.float32)], ids=str)
def test_largest_maps_and_other_calls(levels, C, dtype):
    """Around the most that LDS holds (987 rows of 128 bytes); one distribution for all heads, packed; stage 2 with scores and plain."""
    from dfa3D import _ext, _lib
    S = sum(h * w for h, w in levels)
    t = _as_inputs(tiny_case(seed=S, B=2, M=4, C=C, D=8, Q=32 * S // 8 + 57, P=8 // len(levels), levels=levels))
    value, dist, sh, lsi, loc, attn = _on(_dev(), t, dtype)
    value[0, S // 2, 1] = float("nan")                     # reaches the points around it and no others
    one = dist[:, :, :1].contiguous()
    packed = _ext.pack_shared_dist(one, sh, lsi)
    score = _ext.ms_depth_score_sample_forward(dist, sh, lsi, loc, 64)
    sh2, loc2 = sh[:, :2].contiguous(), loc[..., :2].contiguous()

    def all_calls():
        out = list(_ext.dfa3d_fused_forward(value, dist, sh, lsi, loc, attn, 64, need_depth_score=True))
        out += _ext.dfa3d_fused_forward(value, one, sh, lsi, loc, attn, 64, need_depth_score=False, need_weight_update=True, packed_dist=packed)
        out.append(_ext.wms_deform_attn_forward(value, sh2, lsi, loc2, attn, score, 64))
        out.append(_ext.ms_deform_attn_forward(value, sh2, lsi, loc2, attn, 64))
        return [o for o in out if o is not None]
    got = all_calls()
    with _lib.launch_options(iters=2):
        want = all_calls()
    assert len(got) == len(want) >= 5
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=0, atol=0, equal_nan=True)
    assert 0 < got[0].isnan().any(-1).sum() < got[0].shape[1]
