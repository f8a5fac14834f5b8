"""Level tables with a depth extent: every kind of number that a tensor is filled with."""
import numpy as np
import pytest
import torch

from dfa3D.modules import MSDeformableAttention3D_DFA3D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth", [7, -1, 0, True, np.int64(7), np.int32(5), 7.0, 2 ** 31 - 1, 2 ** 31, 2 ** 40 + 3, -2 ** 31, -2 ** 31 - 1,
                                   torch.tensor(9)], ids=lambda d: f"{type(d).__name__} {d}")
def test_depth_of_any_kind(depth):
    shapes = torch.tensor([[6, 9], [3, 5]])
    want = torch.tensor([[6, 9, int(depth)], [3, 5, int(depth)]])
    got = MSDeformableAttention3D_DFA3D.get_spatial_shape_3D(shapes.cuda(), depth)
    assert got.is_cuda and got.is_contiguous() and torch.equal(got.cpu(), want)
    assert torch.equal(MSDeformableAttention3D_DFA3D.get_spatial_shape_3D(shapes, depth), want)
