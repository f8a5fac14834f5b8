"""Depth taps of a part of the points by scalar loads (large maps, whose coarser levels are in LDS or not): the scores are those of the kernel of stage 1, which
takes them all by vector loads, to the bit, and the sums those of stage 2 with them, but for their order.  Units of one to more points than a wavefront has lanes, few and odd bins, a distribution that begins
between two cache lines, locations outside the map and the depth range, levels that do not fit the keys, and numbers that are none."""
import pytest
import torch

from test_gpu_parity import F32_FWD

pytestmark = pytest.mark.gpu


PYRAMID = ((116, 120), (58, 60), (29, 30), (15, 15))


@pytest.mark.parametrize("levels,M,C,D,P,Q", [
    (PYRAMID, 8, 32, 64, 8, 5101),                         # 32 points a unit: four of them
    (PYRAMID, 8, 4, 129, 2, 20003),
    (PYRAMID, 2, 16, 111, 3, 53401),                       # 12 points: one; bins at odd places
    (PYRAMID, 4, 8, 97, 17, 4803),                         # 68 points: two rounds
    (((160, 190), (80, 95), (40, 48), (20, 24)), 8, 48, 2, 4, 10003),     # two bins
    (PYRAMID[:2] + PYRAMID[:1:-1], 8, 32, 64, 8, 5101),    # no pyramid
    (((116, 200), (58, 100), (29, 50)), 4, 32, 64, 4, 321),               # 2-byte elements: three sixteenths from 5 MB on
    (((116, 200), (58, 100), (29, 50)), 2, 60, 91, 8, 43),
    # all rows from memory, an eighth of a unit's points (3.5 MB and more) and three sixteenths (6 MB and more)
    (PYRAMID, 3, 32, 64, 8, 70), (PYRAMID, 2, 5, 64, 5, 33), (PYRAMID[:1], 2, 64, 33, 3, 130), (PYRAMID[:1], 1, 72, 60, 1, 7), (PYRAMID[:1], 2, 8, 97, 4, 9),
    (PYRAMID[:2], 5, 16, 77, 1, 31), (PYRAMID[:2], 2, 130, 6, 70, 5), (PYRAMID, 8, 12, 101, 2, 1), (PYRAMID[:1], 2, 64, 33, 90, 11),
], ids=str)
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_same_taps_as_stage_1(levels, M, C, D, P, Q, shared, dtype):
    from dfa3D import _ext
    torch.manual_seed(Q)
    dev, B, L = "cuda", 2, len(levels)
    S = sum(h * w for h, w in levels)
    n = B * S * (1 if shared else M) * D
    value = torch.randn(B, S, M, C, device=dev).to(dtype)
    by = 1 if dtype == torch.float32 or D % 2 else 2       # (2-byte bins at odd places are not taken by words)
    dist = torch.rand(n + by, device=dev).to(dtype)[by:].view(B, S, 1 if shared else M, D)
    sh = torch.tensor([[h, w, D] for h, w in levels], device=dev)
    starts = [sum(h * w for h, w in levels[:l]) for l in range(L)]
    lsi = torch.tensor(starts, device=dev)
    loc = torch.rand(B, Q, M, L, P, 3, device=dev) * 1.3 - 0.15
    loc[0, Q - 1, 0, 0, 0] = float("nan")
    loc[1, Q // 2, M - 1, L - 1, P - 1, 2] = float("inf")
    attn = torch.rand(B, Q, M, L, P, device=dev)
    dist[1, S - 1, -1, -1] = float("nan")                  # the last number of all
    dist[0, 0, 0, 0] = float("inf")
    for bad in (False, True):
        if bad:                                            # a level that does not fit the keys is none
            sh = sh.clone()
            sh[L - 1, 0] += 50
        got = _ext.dfa3d_fused_forward(value, dist, sh, lsi, loc, attn, 64, need_depth_score=True, need_weight_update=True)
        want = _ext.ms_depth_score_sample_forward(dist.expand(B, S, M, D).contiguous(), sh, lsi, loc, 64)
        bits = torch.int32 if dtype == torch.float32 else torch.int16
        assert torch.equal(got[1].view(bits), want.view(bits))
        # stage 2 with the scores as they are stored; a 2-byte score is rounded there, and the sum once more
        out = _ext.wms_deform_attn_forward(value, sh[:, :2].contiguous(), lsi, loc[..., :2].contiguous(), attn, want, 64)
        update = (want.double().mean(-1) * attn).sum((-1, -2)).float()
        tol = F32_FWD if dtype == torch.float32 else dict(rtol=2 ** -7, atol=2 ** -8 * float(attn.sum((-1, -2)).max()) * 4)
        torch.testing.assert_close(got[0].float(), out.float(), **tol, equal_nan=True)
        torch.testing.assert_close(got[2].view(update.shape), update, **tol, equal_nan=True)
