"""Backwards with few points, which go to the direct kernels: where the line lies, gradients on both sides of it against the tile kernels',
and the tile kernels at sizes that the line gives to the others."""
import ctypes

import pytest
import torch

from dfa3D import _ext, _lib


def _options(**fields):
    return ctypes.pointer(_lib.LaunchOptions(**fields))


def test_line():
    """Scratch that a call asks for: none below the line (bfloat16 gradients: their float sums), the tile kernels' above it."""
    L, few = _lib.lib(), _lib.DFA3D_FEW_POINTS

    def fused(Q, heads, code, **fields):
        return L.dfa3d_fused_backward_workspace_bytes(2, 3000, 8, 32, 64, 2, Q, 8, heads, code, _options(**fields))

    for heads in (8, 1):
        tiles = [fused(Q, heads, _lib.DFA3D_F32) for Q in (100, 4000)]
        assert fused(100, heads, _lib.DFA3D_F32, direct=few) == 0 < tiles[0]
        assert fused(4000, heads, _lib.DFA3D_F32, direct=few) == tiles[1] > 0
        assert fused(4000, heads, _lib.DFA3D_F32, direct=1) == fused(4000, heads, _lib.DFA3D_F32, direct=-3) == 0
        assert fused(100, heads, _lib.DFA3D_BF16G, direct=few) >= 4 * 2 * 3000 * (8 * 32 + heads * 64)
        assert fused(100, heads, _lib.DFA3D_BF16G, direct=1) == 0
    assert fused(4000, 8, _lib.DFA3D_F64, direct=few) == 0
    assert L.dfa3d_fused_backward_workspace_bytes(2, 3000, 8, 32, 63, 2, 100, 8, 8, _lib.DFA3D_BF16G, _options(direct=few)) == 0
    plain = lambda Q, **o: L.dfa3d_wms_deform_attn_backward_workspace_bytes(2, 3000, 8, 32, 2, Q, 8, _lib.DFA3D_F32, _options(**o))
    stage1 = lambda Q, **o: L.dfa3d_ms_depth_score_sample_backward_workspace_bytes(2, 3000, 8, 64, 2, Q, 8, _lib.DFA3D_F32, _options(**o))
    for call in (plain, stage1):
        assert call(100, direct=few) == 0 < call(100) and call(8000, direct=few) == call(8000) > 0


def _operands(dev, dtype, C, D, Q, heads, maps=((23, 31), (5, 16)), M=4, P=3):
    g = torch.Generator().manual_seed(C + D + Q)
    S, n = sum(h * w for h, w in maps), len(maps)
    loc = torch.rand(2, Q, M, n, P, 3, generator=g) * 1.2 - 0.1
    loc[0, 0, 0, 0, 0] = torch.tensor([float("nan"), 0.5, 0.5])
    loc[-1, -1, -1, -1, -1] = torch.tensor([0.5, 0.5, float("inf")])
    t = [torch.randn(2, S, M, C, generator=g).to(dev, dtype), torch.randn(2, S, heads, D, generator=g).softmax(-1).to(dev, dtype),
         torch.tensor([[h, w, D] for h, w in maps], device=dev), torch.tensor([0, maps[0][0] * maps[0][1]], device=dev), loc.to(dev),
         torch.rand(2, Q, M, n, P, generator=g).to(dev)]
    return t, torch.randn(2, Q, M * C, generator=g).to(dev, dtype), torch.randn(2, Q, M, n, P, 4, generator=g).to(dev, dtype), \
        torch.randn(2, Q, M, 1, generator=g).to(dev)


def _all_gradients(t, go, g_score, g_wu):
    value, dist, shapes, start, loc, attn = t
    xy, shapes2 = loc[..., :2].contiguous(), shapes[:, :2].contiguous()
    got = {"fused": _ext.dfa3d_fused_gradients(*t, go, None, 64, grad_weight_update=g_wu),
           "scores arriving": _ext.dfa3d_fused_gradients(*t, go, g_score, 64),
           "plain": _ext.attention_gradients(value, shapes2, start, xy, attn, None, go, 64)[:3],
           "stage 2": _ext.attention_gradients(value, shapes2, start, xy, attn, g_score.abs(), go, 64)}
    if dist.shape[2] == value.shape[2]:
        got["stage 1"] = _ext.depth_score_gradients(dist, shapes, start, loc, g_score, 64)
    return got


@pytest.mark.gpu
@pytest.mark.parametrize("C,D,Q,heads", [(4, 4, 1, 4), (32, 64, 40, 4), (32, 64, 40, 1), (20, 59, 333, 4), (64, 16, 7, 1), (68, 8, 50, 4), (32, 1, 90, 4),
                                         (32, 16, 3000, 4), (32, 16, 3000, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gradients_of_both_kinds_of_kernels(dtype, C, D, Q, heads):
    """The direct kernels' sums are those of the tile kernels in another order: a few roundings of float; in bfloat16 one
    rounding of 2^-9 on each side (the tile kernels add theirs in bfloat16 on the rims of tiles, up to four times)."""
    dev = torch.device("cuda:0")
    operands = _operands(dev, dtype, C, D, Q, heads)
    by_size = _all_gradients(*operands)
    with _lib.launch_options(chunk=0):                        # options in force: the tile kernels
        tiles = _all_gradients(*operands)
    for kind, got in by_size.items():
        for i, (a, b) in enumerate(zip(got, tiles[kind])):
            assert a.dtype == b.dtype and a.shape == b.shape and torch.isfinite(a).all(), (kind, i)
            scale = b.double().norm().clamp(min=1e-30)
            assert ((a.double() - b.double()).norm() / scale).item() < (2e-6 if a.dtype == torch.float32 else 5 * 2.0 ** -9), (kind, i)


@pytest.mark.gpu
def test_infinite_gradient_on_a_zero_weight():
    """0 * inf arrives as NaN from either kind of kernels, at the same places."""
    dev = torch.device("cuda:0")
    t, go, _, _ = _operands(dev, torch.float32, 32, 16, 20, 4)
    t[4].nan_to_num_(0.5, 0.5)
    t[5][:, ::2] = 0
    go[0, 4, 3] = go[1, 7, 40] = float("inf")
    got = _ext.dfa3d_fused_gradients(*t, go, None, 64)
    with _lib.launch_options(chunk=0):
        want = _ext.dfa3d_fused_gradients(*t, go, None, 64)
    assert want[0].isnan().any()
    for a, b in zip(got, want):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf())


@pytest.mark.gpu
@pytest.mark.parametrize("module,test,args", [
    ("test_gpu_no_bins", "test_more_tiles_than_counters", (32, 64, 3)), ("test_gpu_no_bins", "test_more_tiles_than_counters", (96, 16, 3)),
    ("test_gpu_no_bins", "test_gradients_arriving_at_every_output", ()),
    ("test_gpu_shared_keys", "test_float32_gradients", (32, 64)), ("test_gpu_shared_keys", "test_float32_gradients", (96, 41)),
    ("test_gpu_shared_keys", "test_bfloat16_gradients", (32, 64, "per-head")), ("test_gpu_shared_keys", "test_bfloat16_gradients", (32, 64, "shared")),
    ("test_gpu_many_batches", "test_gradients_of_every_batch_element_and_head", (65600, 2, 4))], ids=lambda v: "")
def test_tile_kernels_below_the_line(oracle, module, test, args):
    """Tests of the tile kernels that call the Functions with few points, once more with launch options in force."""
    import importlib
    with _lib.launch_options(chunk=0):
        getattr(importlib.import_module(module), test)(oracle, *args)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,C,D,skip", [(torch.float32, 32, 9, 3), (torch.float32, 64, 16, 2), (torch.bfloat16, 44, 8, 5), (torch.bfloat16, 32, 16, 2)])
def test_tile_kernels_below_the_line_on_views(dtype, C, D, skip):
    import test_gpu_offset_views as views
    with _lib.launch_options(chunk=0):
        for run in (views._one_stage, views._two_stage):
            views.test_views_off_every_boundary(run, dtype, C, D, skip)
