"""Tile kernel, rows shorter than their lane group: the grad_out rows come to LDS in whole 16-byte pieces or, where a row ends within
one, by registers.  What lies in LDS beyond a row's channels must not count, whatever was there before."""
import pytest
import torch

from test_gpu_cell_walk import _inputs
from test_gpu_parity import _assert_per_point_within_term_count_bound, _assert_sums_within_term_count_bound, _dev

pytestmark = pytest.mark.gpu


def _backward(inp, dev, dtype):
    from dfa3D import _ext
    t = {k: v.to(dev) for k, v in inp.items()}
    value, dist, go = (t[k].to(dtype) for k in ("value", "value_dpt_dist", "grad_output"))
    gv, gd = torch.zeros(value.shape, device=dev), torch.zeros(dist.shape, device=dev)
    gl, ga = torch.empty_like(t["sampling_locations"]), torch.empty_like(t["attention_weights"])
    _ext.dfa3d_fused_backward(value, dist, t["spatial_shapes"], t["level_start_index"], t["sampling_locations"], t["attention_weights"],
                              go, None, gv, gd, gl, ga, 64)
    return gv.cpu(), gd.cpu(), gl.cpu(), ga.cpu()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C", [4, 8, 12, 20, 24, 28, 36, 40, 44, 48, 52, 56, 60])
def test_short_rows_after_rows_of_nan(oracle, C, dtype):
    """Every workgroup of the launch before leaves NaN in all of its staged rows, which lie where this launch's do."""
    dev, D = _dev(), 16
    full = 16 if C <= 16 else 32 if C <= 32 else 64
    before = _inputs(full, D, H=160, W=160, M=4)             # more work items than workgroups
    _backward(dict(before, grad_output=torch.full_like(before["grad_output"], float("nan"))), dev, dtype)
    inp = _inputs(C, D, H=29, W=37)
    gv, gd, gl, ga = _backward(inp, dev, dtype)
    out, score = oracle.dfa3d_forward(*(inp[k] for k in ("value", "value_dpt_dist", "spatial_shapes", "level_start_index",
                                                          "sampling_locations", "attention_weights")))
    _assert_per_point_within_term_count_bound(oracle, inp, out, score, gl, ga)
    _assert_sums_within_term_count_bound(oracle, inp, gv, gd)
