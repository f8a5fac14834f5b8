"""Operands that are contiguous views into larger buffers and start on no wider boundary than an element's: the same results as from
buffers of their own (every kernel reads them with wide loads, the tile kernels also straight into LDS)."""
import pytest
import torch

from dfa3D import functional as f
from test_gpu_parity import _dev

pytestmark = pytest.mark.gpu


def _inputs(C, D, dtype, dev, Q=700, M=4, P=4, maps=((23, 31), (12, 16))):
    g = torch.Generator().manual_seed(C + D)
    S = sum(h * w for h, w in maps)
    return {"value": torch.randn(2, S, M, C, generator=g).to(dev, dtype),
            "dist": torch.randn(2, S, M, D, generator=g).softmax(-1).to(dev, dtype),
            "loc": (torch.rand(2, Q, M, len(maps), P, 3, generator=g) * 1.1 - 0.05).to(dev),
            "attn": torch.rand(2, Q, M, len(maps), P, generator=g).to(dev),
            "go": torch.randn(2, Q, M * C, generator=g).to(dev, dtype)}, \
        torch.tensor([[h, w, D] for h, w in maps], device=dev), torch.tensor([0, maps[0][0] * maps[0][1]], device=dev)


def _view(t, skip):
    """The same numbers `skip` elements into a buffer whose other elements are NaN."""
    whole = torch.full((t.numel() + skip + 8,), float("nan"), dtype=t.dtype, device=t.device)
    part = whole[skip:skip + t.numel()].view(t.shape)
    part.copy_(t)
    assert part.is_contiguous() and (skip == 0 or part.data_ptr() % 16 != 0)
    return part


def _one_stage(t, shapes, start):
    out, score = f.MultiScale3DDeformableAttnFunction.apply(t["value"], t["dist"], shapes, start, t["loc"], t["attn"], 64)
    return (out, score) + torch.autograd.grad(out, [t[k] for k in ("value", "dist", "loc", "attn")], t["go"])


def _two_stage(t, shapes, start):
    score = f.MultiScaleDepthScoreSampleFunction.apply(t["dist"], shapes, start, t["loc"], 64)
    out = f.WeightedMultiScaleDeformableAttnFunction.apply(t["value"], shapes[:, :2].contiguous(), start, t["loc"][..., :2].contiguous(),
                                                           t["attn"], score, 64)
    return (out, score) + torch.autograd.grad(out, [t[k] for k in ("value", "dist", "loc", "attn")], t["go"])


@pytest.mark.parametrize("run", [_one_stage, _two_stage])
@pytest.mark.parametrize("dtype,C,D,skip", [(torch.float32, 20, 16, 1), (torch.float32, 32, 9, 3), (torch.float32, 64, 16, 2), (torch.float32, 100, 8, 1),
                                            (torch.bfloat16, 24, 16, 1), (torch.bfloat16, 32, 9, 3), (torch.bfloat16, 32, 16, 2),
                                            (torch.bfloat16, 44, 8, 5), (torch.bfloat16, 64, 16, 1), (torch.bfloat16, 72, 8, 1)])
def test_views_off_every_boundary(run, dtype, C, D, skip):
    operands, shapes, start = _inputs(C, D, dtype, _dev())
    results = [run({k: _view(v, n).requires_grad_(k != "go") for k, v in operands.items()}, shapes, start) for n in (0, skip)]
    for name, a, b in zip(("out", "score", "value", "dist", "loc", "attn"), *results):
        # sums in another order, and in bfloat16 what that moves across a rounding boundary
        tol = dict(rtol=2e-5, atol=2e-5) if b.dtype == torch.float32 else dict(rtol=2 ** -6, atol=2 ** -6)
        torch.testing.assert_close(b, a, msg=lambda m, name=name: f"{name}: {m}", **tol)
