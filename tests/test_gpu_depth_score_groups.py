"""Stage 1 forward: blocks of one level and of all levels, of 256 and of 1024 points (four at a time per lane, and the rest), and
points per level that divide neither."""
import pytest
import torch

from forms import tiny_case
from test_gpu_parity import F32_FWD, _as_inputs, _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,M,Q,P,levels", [
    (2, 3, 70, 3, ((9, 14), (5, 7))), (2, 3, 70, 5, ((9, 14), (5, 7), (3, 3))), (1, 2, 5, 300, ((9, 14),)),
    (1, 1, 2, 1500, ((9, 14), (4, 4))),
    (2, 8, 9001, 8, ((21, 30), (11, 15), (6, 8), (3, 4))), (1, 6, 52001, 7, ((21, 30), (11, 15))), (3, 8, 60001, 3, ((21, 30),)),      # over 2^22 points
], ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_scores(oracle, B, M, Q, P, levels, dtype):
    from dfa3D import _ext
    dev = _dev()
    t = _as_inputs(tiny_case(seed=60 + P, B=B, M=M, C=1, D=9, Q=Q, P=P, levels=levels))
    dist, loc = t["value_dpt_dist"].to(dtype), t["sampling_locations"].float().contiguous()
    got = _ext.ms_depth_score_sample_forward(dist.to(dev), t["spatial_shapes"].to(dev), t["level_start_index"].to(dev), loc.to(dev), 64)
    assert torch.isfinite(got).all()
    # a block's first and last queries and some between are compared
    some = torch.unique(torch.cat([torch.arange(min(Q, 40)), torch.arange(max(Q - 40, 0), Q), torch.arange(0, Q, max(Q // 97, 1))]))
    with oracle.float_geometry():
        want = oracle.depth_score_forward(dist.double(), t["spatial_shapes"], t["level_start_index"], loc[:, some].double().contiguous())
    tol = F32_FWD if dtype == torch.float32 else dict(rtol=2.0 ** -8, atol=1e-5)       # stored in bfloat16: one rounding
    torch.testing.assert_close(got[:, some.to(dev)].cpu().double(), want, **tol)
