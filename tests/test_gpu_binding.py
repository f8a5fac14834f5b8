"""The short way of a call (the binding module) against the long way through ctypes: same results from every Function, same
complaint where an operand is not what the kernels read, and the caller's stream."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from forms import tiny_case
from test_gpu_parity import _as_inputs, _dev

pytestmark = pytest.mark.gpu


def _operands(dtype, heads=4, one=False):
    dev = _dev()
    t = _as_inputs(tiny_case(seed=7, B=2, M=heads, C=12, D=6, Q=150, P=3, levels=((9, 11), (5, 6))))
    aux = torch.float32 if dtype == torch.bfloat16 else dtype
    dist = t["value_dpt_dist"].to(dtype).to(dev)
    return dict(value=t["value"].to(dtype).to(dev), dist=dist[:, :, :1].contiguous() if one else dist, shapes=t["spatial_shapes"].to(dev),
                starts=t["level_start_index"].to(dev), loc=t["sampling_locations"].to(aux).to(dev), attn=t["attention_weights"].to(aux).to(dev))


def _run(o, kind):
    from dfa3D import functional as f
    leaves = [o[k].detach().requires_grad_() for k in ("value", "dist", "loc", "attn")]
    value, dist, loc, attn = leaves
    sh, st = o["shapes"], o["starts"]
    g = torch.Generator(device=value.device).manual_seed(3)
    if kind == "one_stage":
        out = f.MultiScale3DDeformableAttnFunction.apply(value, dist, sh, st, loc, attn, 64)
    elif kind == "stage_1":
        out, leaves = (f.MultiScaleDepthScoreSampleFunction.apply(dist, sh, st, loc, 64),), [dist, loc]
    elif kind == "weight_update":
        out = f.MultiScale3DDeformableAttnWeightUpdateFunction.apply(value, dist, sh, st, loc, attn, 64)
    else:
        loc2, sh2 = loc.detach()[..., :2].contiguous().requires_grad_(), sh[:, :2].contiguous()
        leaves[2] = loc2
        if kind == "plain":
            out = (f.MultiScaleDeformableAttnFunction.apply(value, sh2, st, loc2, attn, 64),)
            leaves = [value, loc2, attn]
        else:
            score = torch.rand(*loc.shape[:5], 4, generator=g, device=value.device).to(value.dtype).requires_grad_()
            out = (f.WeightedMultiScaleDeformableAttnFunction.apply(value, sh2, st, loc2, attn, score, 64),)
            leaves = [value, loc2, attn, score]
    grads = [torch.randn(x.shape, generator=g, device=x.device).to(x.dtype) for x in out]
    return [x.detach() for x in out] + list(torch.autograd.grad(out, leaves, grads))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16], ids=["fp32", "fp64", "bf16"])
@pytest.mark.parametrize("kind", ["one_stage", "weight_update", "weight_update_one", "stage_1", "stage_2", "plain"])
def test_both_ways(monkeypatch, kind, dtype):
    from dfa3D import _ext, _lib

    class Watched:
        """The binding module; notes what was called and whether it took the call."""
        def __init__(self):
            self.took = {}

        def __getattr__(self, name):
            call = getattr(_lib.binding(), name)

            def watched(*args):
                got = call(*args)
                self.took[name] = self.took.get(name, True) and got is not None
                return got
            return watched
    watched, here = Watched(), _ext._here
    monkeypatch.setattr(_ext, "_here", lambda value: (watched, *here(value)[1:]))
    one = kind == "weight_update_one"
    o = _operands(dtype, one=one)
    kind = kind.replace("_one", "") if kind == "weight_update_one" else kind
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        short = _run(o, kind)
    torch.cuda.current_stream().wait_stream(side)
    names = {"stage_1": ("score_forward", "score_gradients"), "one_stage": ("fused_forward", "fused_gradients"),
             "weight_update": ("fused_forward", "fused_gradients")}.get(kind, ("attention_forward", "attention_gradients"))
    assert all(watched.took.get(n) for n in names) and all(took for n, took in watched.took.items() if n != "pack_dist")
    if one and dtype != torch.float64:
        assert watched.took["pack_dist"]
    monkeypatch.setattr(_ext, "_here", lambda value: None)
    long = _run(o, kind)
    assert len(short) == len(long)
    outputs = 1 if kind in ("stage_1", "stage_2", "plain") else 2
    # gradients are added up atomically in no fixed order: a few hundred terms per element
    tol = {torch.float32: dict(rtol=1e-5, atol=1e-4), torch.float64: dict(rtol=1e-12, atol=1e-12), torch.bfloat16: dict(rtol=2 ** -6, atol=1e-2)}[dtype]
    for i, (a, b) in enumerate(zip(short, long)):
        assert a.dtype == b.dtype and a.shape == b.shape
        if i < outputs:
            assert torch.equal(a, b)                                        # no atomics
        else:
            torch.testing.assert_close(a, b, **tol)


def _strided(t):
    return t.transpose(0, 1).contiguous().transpose(0, 1)


@pytest.mark.parametrize("name,spoil", [("value", _strided), ("loc", lambda t: t.double()), ("attn", lambda t: t[:, :-1].contiguous()), ("dist", lambda t: t.cpu()),
                                        ("shapes", lambda t: t.int()), ("starts", lambda t: t[:1].contiguous()), ("value", lambda t: t.half()),
                                        ("dist", lambda t: t[:, :, :2].contiguous())])
def test_same_complaint(monkeypatch, name, spoil):
    from dfa3D import _ext
    o = _operands(torch.float32)
    o[name] = spoil(o[name])
    said = []
    for short in (True, False):
        if not short:
            monkeypatch.setattr(_ext, "_here", lambda value: None)
        with pytest.raises((RuntimeError, TypeError)) as e:
            _ext.dfa3d_fused_forward(o["value"], o["dist"], o["shapes"], o["starts"], o["loc"], o["attn"], 64)
        said.append((type(e.value), str(e.value)))
    assert said[0] == said[1]


def test_subclasses_and_transforms_take_the_long_way():
    from dfa3D import _ext, _lib

    class Own(torch.Tensor):
        pass
    o = _operands(torch.float32)
    native, at, stream = _ext._here(o["value"])
    args = lambda v: (at, stream, v, o["dist"], o["shapes"], o["starts"], o["loc"], o["attn"], 64, True, False, None)
    assert native.fused_forward(*args(o["value"])) is not None
    assert native.fused_forward(*args(torch.nn.Parameter(o["value"]))) is not None
    assert native.fused_forward(*args(o["value"].as_subclass(Own))) is None
    assert native.fused_forward(*args(torch._neg_view(o["value"]))) is None
    seen = []
    torch.func.vmap(lambda v: (seen.append(native.fused_forward(*args(v))), v)[1])(o["value"][None])
    assert seen == [None]
    torch.func.vmap(lambda v: (seen.append(native.fused_forward(*args(o["value"]))), v)[1])(o["value"][None])
    with TorchDispatchMode():
        seen.append(native.fused_forward(*args(o["value"])))
    with FakeTensorMode():
        seen.append(native.fused_forward(*args(o["value"])))
    assert seen == [None] * 4
    with _lib.launch_options(iters=2):
        assert _ext._here(o["value"]) is None
