"""Forward with value rows in LDS, of all of a small map or of a pyramid's coarser levels: row lengths on both sides of every lane
group, points per unit from one to more than a wavefront holds, a last share of the queries that is not full, and maps on both sides
of what LDS holds.  Walking several groups per wavefront on request (iters = 2) keeps the gathers from memory, which for a whole map form
the same sums in the same order."""
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


@pytest.mark.parametrize("levels,M,C,P,dtype", [
    (((40, 50), (20, 25), (10, 13)), 8, 32, 4, torch.float32),       # two of three levels fit
    (((40, 50), (20, 25), (10, 13)), 4, 20, 5, torch.float32),
    (((56, 60), (28, 30), (14, 15), (7, 8)), 8, 32, 3, torch.bfloat16),
    (((56, 60), (28, 30), (14, 15), (7, 8)), 2, 64, 17, torch.float32),        # two rounds of 64 points per unit
    (((30, 40), (15, 20), (8, 10)), 8, 32, 4, torch.float32),       # (the finest level just does not fit)
    (((20, 25), (40, 50), (10, 13)), 8, 32, 4, torch.float32),      # no pyramid: the last level alone fits
    (((13, 13), (20, 25), (40, 50)), 8, 32, 4, torch.float32),      # coarse to fine: none does
], ids=str)
def test_coarser_levels(levels, M, C, P, dtype):
    from dfa3D import _ext, _lib
    L, S = len(levels), sum(h * w for h, w in levels)
    Q = 256 // M * 2200 // P + 29                             # enough points for one workgroup per CU
    t = _as_inputs(tiny_case(seed=S + P, B=1, M=M, C=C, D=5, Q=Q, P=P, levels=levels))
    value, dist, sh, lsi, loc, attn = _on(_dev(), t, dtype)
    value[0, S - 2, 1] = float("nan")
    sh[0, 1] += 10 ** 6 if L == 4 and M == 2 else 0          # a level that is no level of this map
    one = dist[:, :, :1].contiguous()
    packed = _ext.pack_shared_dist(one, sh, lsi)

    def all_calls():
        out = list(_ext.dfa3d_fused_forward(value, dist, sh, lsi, loc, attn, 64, need_depth_score=True))
        out += _ext.dfa3d_fused_forward(value, one, sh, lsi, loc, attn, 64, need_depth_score=False, need_weight_update=True, packed_dist=packed)
        out.append(_ext.ms_deform_attn_forward(value, sh[:, :2].contiguous(), lsi, loc[..., :2].contiguous(), attn, 64))
        return [o for o in out if o is not None]
    got = all_calls()
    with _lib.launch_options(iters=2):
        want = all_calls()
    # the same products, added up in another order: at most 8 additions in one chain and a few above it, each rounded to 2^-24 of at
    # most the sum of the sizes (|value| < 5, weights of a unit sum to at most 1); bfloat16: one rounding of the result
    tol = dict(rtol=1e-6, atol=4e-6) if dtype == torch.float32 else dict(rtol=2 ** -7, atol=1e-5)
    assert len(got) == len(want) >= 4
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, equal_nan=True, **tol)
    assert got[0].isnan().any()
