"""The stage-1 backward with 256, 512 and 1024 threads per tile, which the points per pixel decide: few points on many tiles to more
points in a tile than threads, tiles of 8 x 8 and 8 x 16 pixels, rows from one bin to more than a wavefront takes at a time."""
import pytest
import torch

from forms import tiny_case
from test_gpu_parity import F32_BWD, _as_inputs, _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [1, 30, 112, 130])
@pytest.mark.parametrize("Q,P,tile", [(40, 4, 0), (200, 4, 0), (700, 4, 0), (700, 4, 816), (1100, 16, 816)],
                         ids=["sparse", "few", "many", "many-wide", "rounds"])
def test_stage_one_backward(oracle, D, Q, P, tile):
    """0.2, 1.1, 3.7 and 23 points per pixel: 256, 512 and 1024 threads, the last with several rounds per tile."""
    from dfa3D import _ext, _lib
    dev = _dev()
    t = _as_inputs(tiny_case(seed=50 + D, B=1, M=2, C=1, D=D, Q=Q, P=P, levels=((25, 41), (13, 36))))
    dist, loc = t["value_dpt_dist"].float(), t["sampling_locations"].float().contiguous()
    go = torch.randn(1, Q, 2, 2, P, 4, generator=torch.Generator().manual_seed(3))
    with oracle.float_geometry():
        want, want_gl = oracle.depth_score_backward(dist.double(), t["spatial_shapes"], t["level_start_index"], loc.double(), go.double())
    gd, gl = torch.full(dist.shape, float("nan"), device=dev), torch.full(loc.shape, float("nan"), device=dev)
    with _lib.launch_options(**({"tile": tile} if tile else {})):
        _ext.ms_depth_score_sample_backward_into(dist.to(dev), t["spatial_shapes"].to(dev), t["level_start_index"].to(dev), loc.to(dev),
                                                 go.to(dev), gd, gl, 64, clear=True)
    # D = 1: all points of four pixels meet in one word, up to n = 64 in the mean, a few times that at most
    torch.testing.assert_close(gd.cpu().double(), want, **F32_BWD)
    torch.testing.assert_close(gl.cpu().double(), want_gl, rtol=1e-4, atol=1e-3)     # z gradient: differences of bins, times D
