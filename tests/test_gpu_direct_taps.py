"""Backward on the kernels that add to device memory: a pair of lanes sends both bins of one point, then of the other, so points in odd
numbers, single points, one to three bins, and units spread over as many wavefronts as there are."""
import pytest
import torch

from forms import tiny_case
from test_gpu_parity import _as_inputs, _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,M,Q,P,C,D,levels", [(1, 1, 1, 1, 4, 2, ((3, 4),)), (2, 3, 37, 3, 5, 1, ((5, 7), (3, 3))), (1, 2, 300, 7, 32, 3, ((6, 9),)),
                                                (2, 8, 130, 1, 20, 17, ((9, 5), (4, 3), (2, 2))), (1, 3, 9, 67, 8, 5, ((7, 7),))], ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["fp32", "fp64"])
def test_direct_backward(oracle, B, M, Q, P, C, D, levels, dtype):
    from dfa3D import _ext, _lib
    dev = _dev()
    t = _as_inputs(tiny_case(seed=11 + Q, B=B, M=M, C=C, D=D, Q=Q, P=P, levels=levels))
    o = [t[k].to(dtype) if t[k].is_floating_point() else t[k] for k in
         ("value", "value_dpt_dist", "spatial_shapes", "level_start_index", "sampling_locations", "attention_weights", "grad_output")]
    _, score = oracle.dfa3d_forward(*o[:6])
    want = oracle.dfa3d_backward(*o[:6], score, o[6])
    with _lib.launch_options(direct=1):
        got = _ext.dfa3d_fused_gradients(*[x.to(dev) for x in o[:6]], o[6].to(dev), None, 64)
    # sums of up to Q P corner terms per element, of size 1 to 10, each rounded to 2^-24 (2^-53) of the running sum
    tol = dict(rtol=1e-4, atol=2e-4) if dtype == torch.float32 else dict(rtol=1e-10, atol=1e-10)
    for a, b in zip(got, want):
        torch.testing.assert_close(a.cpu(), b.to(dtype).view_as(a), **tol)
