"""More batch elements, and more heads, than 16 bits hold: the work items of the tile backward name both."""
import pytest
import torch

from forms import tiny_case
from test_gpu_parity import (F32_BWD, F32_FWD, _as_inputs, _compare, _dev, _gpu_one_stage, _gpu_two_stage, _oracle_one_stage)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C", [4, 68], ids=["cell-owned", "row-owned"])
@pytest.mark.parametrize("B,M", [(65600, 2), (2, 32771), (1, 65537)])
def test_gradients_of_every_batch_element_and_head(oracle, B, M, C):
    """One stage, and the two stages apart (which is the stage-1 tile kernel as well).  Batches go in steps of 64."""
    dev = _dev()
    inp = _as_inputs(tiny_case(seed=71, B=B, M=M, C=C, D=4, Q=1, P=2, levels=((2, 2), (1, 1)), dtype=torch.float32))
    want = _oracle_one_stage(oracle, inp)
    _compare(_gpu_one_stage(inp, dev), want, F32_FWD, F32_BWD)
    _compare(_gpu_two_stage(inp, dev, sliced=True), want, F32_FWD, F32_BWD)
