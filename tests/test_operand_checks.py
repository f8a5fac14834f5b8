"""The checks of the one-kernel entry points take the operands that fit and refuse every other shape and type, whatever order
they look in; runs without a GPU."""
import pytest
import torch

from dfa3D import _ext


def _operands(heads=2, dtype=torch.float32):
    aux = torch.float32 if dtype == torch.bfloat16 else dtype
    return dict(value=torch.zeros(2, 7, 2, 4, dtype=dtype), dist=torch.zeros(2, 7, heads, 5, dtype=dtype),
                shapes3=torch.tensor([[2, 3, 5], [1, 1, 5]]), lsi=torch.tensor([0, 6]),
                loc3=torch.zeros(2, 3, 2, 2, 4, 3, dtype=aux), attn=torch.zeros(2, 3, 2, 2, 4, dtype=aux))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16], ids=str)
@pytest.mark.parametrize("heads", [1, 2])
def test_operands_that_fit(heads, dtype):
    assert _ext._fused_dims(**_operands(heads, dtype), name="f") == (2, 7, 2, 4, 5, 2, 3, 4)


@pytest.mark.parametrize("which", ["value", "dist", "shapes3", "lsi", "loc3", "attn"])
def test_operands_that_do_not(which):
    good = _operands()
    t = good[which]
    wrong = [t.to(torch.int32), t.to(torch.float16), t[0], t.unsqueeze(0)]
    wrong += [torch.cat([t, t], d) for d in range(t.dim())
              if (which, d) not in (("value", 3), ("dist", 3))]          # any number of channels, of bins
    for bad in wrong:
        with pytest.raises((RuntimeError, IndexError)):
            _ext._fused_dims(**{**good, which: bad}, name="f")


def test_placement():
    a = torch.zeros(4, 4)
    with pytest.raises(RuntimeError, match="b tensor has to be contiguous"):
        _ext._contig_on_gpu(a=a, b=a.t()[:2])
    with pytest.raises(RuntimeError, match="a must be a CUDA tensor"):
        _ext._contig_on_gpu(a=a, b=a)
