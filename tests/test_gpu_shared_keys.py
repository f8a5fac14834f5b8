"""Levels that share keys (a level table may give one map to several levels): the tiles of two levels then meet on the same
rows of grad_value and grad_dist, and both must arrive.  Every kernel of the tile backward: the cell-owned one in each of
its lane groupings, with bins that are and are no multiple of four, the row-owned one for longer rows, one distribution per
head and one for all heads, float32 and bfloat16 gradients, buffers that hold anything on entry."""
import pytest
import torch

from forms import tiny_case
from test_gpu_parity import (F32_BWD, F32_FWD, _as_inputs, _assert_sums_within_term_count_bound, _dev, _gpu_one_stage,
                             _gpu_two_stage, _oracle_one_stage)

pytestmark = pytest.mark.gpu

LEVELS = ((33, 17), (30, 18), (8, 7))


def _shared_keys_case(C, D, Q=700):
    inp = _as_inputs(tiny_case(seed=60 + C + D, B=2, M=4, C=C, D=D, Q=Q, P=4, levels=LEVELS, dtype=torch.float32))
    inp["level_start_index"] = torch.tensor([0, 7, 100])           # the second starts inside the first one's first row
    return inp


@pytest.mark.parametrize("C,D", [(4, 1), (16, 59), (20, 41), (32, 64), (32, 41), (40, 33), (64, 16), (96, 64), (96, 41), (7, 8)])
def test_float32_gradients(oracle, C, D):
    dev = _dev()
    inp = _shared_keys_case(C, D)
    want = _oracle_one_stage(oracle, inp)
    for got in (_gpu_one_stage(inp, dev), _gpu_two_stage(inp, dev, sliced=True)):
        for i in (0, 1, 4, 5):
            torch.testing.assert_close(got[i], want[i], **(F32_FWD if i < 2 else F32_BWD))
        _assert_sums_within_term_count_bound(oracle, inp, got[2], got[3])


@pytest.mark.parametrize("C,D", [(32, 64), (64, 16)])
@pytest.mark.parametrize("heads", ["per-head", "shared"])
def test_bfloat16_gradients(oracle, C, D, heads):
    from dfa3D.functional import MultiScale3DDeformableAttnFunction
    dev = _dev()
    inp = _shared_keys_case(C, D)
    r16 = dict(inp, **{k: inp[k].bfloat16().float() for k in ("value", "value_dpt_dist", "grad_output")})
    if heads == "shared":
        one = r16["value_dpt_dist"][:, :, :1].contiguous()
        r16["value_dpt_dist"] = one.repeat(1, 1, 4, 1)
    dist = one if heads == "shared" else r16["value_dpt_dist"]
    leaves = [t.to(dev).requires_grad_() for t in (r16["value"].bfloat16(), dist.bfloat16(), inp["sampling_locations"],
                                                   inp["attention_weights"])]
    out, _ = MultiScale3DDeformableAttnFunction.apply(leaves[0], leaves[1], inp["spatial_shapes"].to(dev),
                                                      inp["level_start_index"].to(dev), leaves[2], leaves[3], 64)
    gv, gd, _, _ = torch.autograd.grad(out, leaves, r16["grad_output"].bfloat16().to(dev))
    # a row collects from up to four tiles of each of the three levels: 12 adds that round the stored sum
    _assert_sums_within_term_count_bound(oracle, r16, gv.float().cpu(), gd.float().cpu(), storage_rel=2.0 ** -8,
                                         shared_dist=heads == "shared", atomic_rel=12 * 2.0 ** -9)
