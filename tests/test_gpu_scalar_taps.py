"""Depth taps of a part of the points by scalar loads (large maps whose coarser levels are in LDS): the scores are those of the path that gathers everything
from memory (iters = 2) to the bit, the sums but for their order.  Units of one to more points than a wavefront has lanes, few and odd bins, a distribution that begins
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
], ids=str)
@pytest.mark.parametrize("shared", [False, True])
def test_same_taps_as_from_memory(levels, M, C, D, P, Q, shared):
    from dfa3D import _ext, _lib
    torch.manual_seed(Q)
    dev, B, L = "cuda", 2, len(levels)
    S = sum(h * w for h, w in levels)
    n = B * S * (1 if shared else M) * D
    value = torch.randn(B, S, M, C, device=dev)
    dist = torch.rand(n + 1, device=dev)[1:].view(B, S, 1 if shared else M, D)
    sh = torch.tensor([[h, w, D] for h, w in levels], device=dev)
    starts = [sum(h * w for h, w in levels[:l]) for l in range(L)]
    lsi = torch.tensor(starts, device=dev)
    loc = torch.rand(B, Q, M, L, P, 3, device=dev) * 1.3 - 0.15
    loc[0, 1, 0, 0, 0] = float("nan")
    loc[1, 2, M - 1, L - 1, P - 1, 2] = float("inf")
    attn = torch.rand(B, Q, M, L, P, device=dev)
    dist[1, S - 1, -1, -1] = float("nan")                  # the last number of all
    dist[0, 0, 0, 0] = float("inf")
    for bad in (False, True):
        if bad:                                            # a level that does not fit the keys is none
            sh = sh.clone()
            sh[L - 1, 0] += 50
        got = _ext.dfa3d_fused_forward(value, dist, sh, lsi, loc, attn, 64, need_depth_score=True, need_weight_update=True)
        with _lib.launch_options(iters=2):
            want = _ext.dfa3d_fused_forward(value, dist, sh, lsi, loc, attn, 64, need_depth_score=True, need_weight_update=True)
        assert torch.equal(got[1].view(torch.int32), want[1].view(torch.int32))
        torch.testing.assert_close(got[2], want[2], rtol=0, atol=0, equal_nan=True)
        torch.testing.assert_close(got[0], want[0], **F32_FWD, equal_nan=True)
