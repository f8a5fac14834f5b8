"""The stage-1 backward on tiles: tiles whose points fit one work item (stored pixels) and several (all added), rows that
are no whole 16-byte groups, one bin, many points on one pixel and depth, levels that share keys, and a gradient buffer that
already holds something: it is added to, as the reference does."""
import pytest
import torch

from forms import tiny_case
from test_gpu_parity import F32_BWD, _as_inputs, _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,levels,Q,chunk,where", [
    (64, ((33, 17), (8, 7)), 300, 0, None), (112, ((17, 16), (1, 9)), 200, 0, None), (59, ((9, 23),), 250, 0, None),
    (1, ((16, 15), (4, 4)), 120, 0, None), (128, ((24, 9),), 500, 64, None), (16, ((8, 8), (3, 3)), 900, 0, 0.52),
    (200, ((15, 15),), 100, 0, None), (4, ((40, 41),), 2000, 64, None)])
@pytest.mark.parametrize("overlap", [False, True], ids=["levels", "shared-keys"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_stage_one_backward(oracle, D, levels, Q, chunk, where, overlap, dtype):
    from dfa3D import _ext, _lib
    dev = _dev()
    t = _as_inputs(tiny_case(seed=40 + D, B=2, M=3, C=1, D=D, Q=Q, P=4, levels=levels))
    dist, loc = t["value_dpt_dist"].to(dtype), t["sampling_locations"].float().contiguous()
    if where is not None:
        loc = loc * 0 + where
    sh, lsi = t["spatial_shapes"], t["level_start_index"].clone()
    if overlap:
        lsi.zero_()                              # every level reads and adds to the first keys
    g = torch.Generator().manual_seed(3)
    go = torch.randn(2, Q, 3, len(levels), 4, 4, generator=g).to(dtype)
    held = torch.randn(dist.shape, generator=g)
    with oracle.float_geometry():
        want, want_gl = oracle.depth_score_backward(dist.double(), sh, lsi, loc.double(), go.double())
    gd, gl = held.clone().to(dev), torch.empty(loc.shape, device=dev)
    with _lib.launch_options(**({"chunk": chunk} if chunk else {})):
        _ext.ms_depth_score_sample_backward(dist.to(dev), sh.to(dev), lsi.to(dev), loc.to(dev), go.to(dev), gd, gl, 64)
    # all points on one pixel: n = 4 Q L (16 for the corners) terms in one word, float32 sums in any order are good to about
    # 2^-24 n^(1/2) of their size times the chain's growth n^(1/2)
    tol = F32_BWD if where is None else dict(rtol=1e-4, atol=2.0 ** -24 * 16 * Q * len(levels))
    torch.testing.assert_close((gd.cpu() - held).double(), want, **tol)
    torch.testing.assert_close(gl.cpu().double(), want_gl, rtol=1e-4, atol=1e-3)     # z gradient: differences of bins, times D
    # a buffer that may hold anything
    for direct in (0, 1):
        fresh = torch.full(dist.shape, float("nan"), device=dev)
        with _lib.launch_options(direct=direct, **({"chunk": chunk} if chunk else {})):
            _ext.ms_depth_score_sample_backward_into(dist.to(dev), sh.to(dev), lsi.to(dev), loc.to(dev), go.to(dev), fresh, gl, 64,
                                                     clear=True)
        torch.testing.assert_close(fresh.cpu().double(), want, **tol)
