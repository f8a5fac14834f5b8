"""The forward's split of a wavefront over units and row slots, at the edges of its ranges: points per unit from 1 to more
than a wavefront holds, row lengths on both sides of every row tiling, few queries (units spread over more wavefronts)
and many, a last group of units that is not full."""
import pytest
import torch

from forms import tiny_case
from test_gpu_parity import F32_FWD, _as_inputs, _dev

pytestmark = pytest.mark.gpu

LEVELS = ((9, 13), (5, 7), (3, 4), (2, 2))


@pytest.mark.parametrize("L,P,C,Q", [
    (1, 1, 32, 3001), (1, 2, 16, 1500), (1, 3, 20, 1111), (1, 4, 32, 2049), (1, 4, 3, 7), (1, 5, 24, 901), (1, 8, 32, 640),
    (2, 5, 36, 513), (2, 6, 5, 333), (3, 5, 20, 257), (2, 8, 64, 300), (4, 5, 32, 700), (1, 9, 32, 900), (2, 5, 16, 1301), (1, 10, 130, 77), (3, 7, 40, 129), (4, 8, 32, 260), (4, 8, 32, 3),
    (3, 11, 12, 65), (4, 16, 28, 33), (4, 17, 100, 31), (4, 33, 32, 9), (1, 4, 260, 40), (2, 4, 1, 90), (2, 4, 66, 50)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16], ids=["fp32", "fp64", "bf16"])
def test_units_and_row_slots(oracle, L, P, C, Q, dtype):
    from dfa3D import _ext
    dev = _dev()
    t = _as_inputs(tiny_case(seed=900 + L * P + C, B=2, M=3, C=C, D=7, Q=Q, P=P, levels=LEVELS[:L]))
    store = torch.bfloat16 if dtype == torch.bfloat16 else dtype
    aux = torch.float32 if dtype == torch.bfloat16 else dtype
    value, dist = t["value"].to(store), t["value_dpt_dist"].to(store)
    loc, attn = t["sampling_locations"].to(aux), t["attention_weights"].to(aux)
    sh, lsi = t["spatial_shapes"], t["level_start_index"]
    want, want_score = oracle.dfa3d_forward(value.to(aux), dist.to(aux), sh, lsi, loc, attn)
    got, score, wu = _ext.dfa3d_fused_forward(value.to(dev), dist.to(dev), sh.to(dev), lsi.to(dev), loc.to(dev),
                                              attn.to(dev), 64, need_depth_score=True, need_weight_update=True)
    # bfloat16: the sums are float32, the results rounded once (2^-9 of their size)
    tol = {torch.float32: F32_FWD, torch.float64: dict(rtol=1e-10, atol=1e-11),
           torch.bfloat16: dict(rtol=2 ** -8, atol=1e-5)}[dtype]
    torch.testing.assert_close(got.cpu().to(aux), want, **tol)
    torch.testing.assert_close(score.cpu().to(aux), want_score, **tol)
    want_wu = (want_score.mean(-1) * attn).flatten(-2).sum(-1, keepdim=True)
    torch.testing.assert_close(wu.cpu().to(aux).view_as(want_wu), want_wu, **{**tol, **(F32_FWD if aux == torch.float32 else {})})
