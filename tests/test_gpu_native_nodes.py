"""Calls that the binding module records as a whole: the same gradients as from the Functions' own nodes in Python, and the same answers to
what a graph is asked (saved-tensor hooks, a backward that is recorded, a second one, operands changed in place, compiled autograd)."""
import pytest
import torch
from torch.utils.checkpoint import checkpoint

from dfa3D import functional as f
from forms import tiny_case
from test_gpu_parity import _as_inputs, _dev

pytestmark = pytest.mark.gpu

KINDS = {"score": f.MultiScaleDepthScoreSampleFunction, "stage2": f.WeightedMultiScaleDeformableAttnFunction, "plain": f.MultiScaleDeformableAttnFunction,
         "fused": f.MultiScale3DDeformableAttnFunction, "weight_update": f.MultiScale3DDeformableAttnWeightUpdateFunction}


def _args(kind, dtype=torch.float32, one=False):
    dev = _dev()
    t = _as_inputs(tiny_case(seed=5, B=2, M=4, C=12, D=6, Q=60, P=3, levels=((9, 11), (5, 6))))
    aux = torch.float32 if dtype == torch.bfloat16 else dtype
    value, dist = (t[k].to(dev, dtype) for k in ("value", "value_dpt_dist"))
    if one:
        dist = dist[:, :, :1].contiguous()
    loc, attn = (t[k].to(dev, aux) for k in ("sampling_locations", "attention_weights"))
    s3, start = t["spatial_shapes"].to(dev), t["level_start_index"].to(dev)
    s2, xy = s3[:, :2].contiguous(), loc[..., :2].contiguous()
    if kind == "score":
        return [dist, s3, start, loc, 64]
    if kind == "stage2":
        return [value, s2, start, xy, attn, torch.rand(*attn.shape, 4, device=dev).to(dtype), 64]
    return [value, s2, start, xy, attn, 64] if kind == "plain" else [value, dist, s3, start, loc, attn, 64]


def _record(kind, args):
    args = [a.detach().clone().requires_grad_(a.is_floating_point()) if torch.is_tensor(a) else a for a in args]
    out = KINDS[kind].apply(*args)
    return (out if isinstance(out, tuple) else (out,)), [a for a in args if torch.is_tensor(a) and a.requires_grad]


def _upstream(out, seed=0):
    g = torch.Generator(device=out[0].device).manual_seed(seed)
    return [torch.randn(o.shape, generator=g, device=o.device).to(o.dtype) for o in out]


def _is_native(out):
    return "CppNode<dfa3d::" in out.grad_fn.name()


def _close(a, b):
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and x.shape == y.shape
        tol = {torch.float32: 2e-6, torch.float64: 1e-14, torch.bfloat16: 2.0 ** -8}[x.dtype]      # atomics in any order; a rounding of what is stored
        assert (x.double() - y.double()).norm() <= tol * y.double().norm().clamp(min=1e-30)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64])
@pytest.mark.parametrize("kind,one", [("score", False), ("stage2", False), ("plain", False), ("fused", False), ("fused", True), ("weight_update", False),
                                      ("weight_update", True)])
def test_same_results_as_a_python_node(monkeypatch, kind, one, dtype):
    args = _args(kind, dtype, one)
    results = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(KINDS[kind], "kind", None)
        out, leaves = _record(kind, args)
        assert _is_native(out[0]) == native and all(o.requires_grad for o in out)
        grads = torch.autograd.grad(out, leaves, _upstream(out), retain_graph=True)
        each = [torch.autograd.grad(o, leaves, g, retain_graph=True, allow_unused=True) for o, g in zip(out, _upstream(out, 1))]
        # incoming gradients that are neither contiguous nor of the output's type
        odd = [g.transpose(0, 1).contiguous().transpose(0, 1) for g in _upstream(out, 2)]
        again = torch.autograd.grad(out, leaves, odd)
        results.append([o.detach() for o in out] + [g for gs in (grads, *each, again) for g in gs])
    assert len(results[0]) == len(results[1])
    _close(*results)


@pytest.mark.parametrize("kind", KINDS)
def test_what_a_graph_is_asked(kind):
    args = _args(kind)
    out, leaves = _record(kind, args)
    up = _upstream(out)
    want = torch.autograd.grad(out, leaves, up, retain_graph=True)
    # a backward that is recorded gives the same numbers, and is refused when it is asked for its own gradient
    some = torch.autograd.grad(out, leaves, [u.clone().requires_grad_() for u in up], create_graph=True)
    _close(some, want)
    with pytest.raises(RuntimeError, match="once_differentiable"):
        some[0].sum().backward()
    _close(torch.autograd.grad(out, leaves, up), want)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, leaves, up)
    # hooks see every tensor that is saved, and what they give back is used
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.cpu(), lambda t: t.to(_dev())):
        out, leaves = _record(kind, args)
    assert _is_native(out[0]) and len(packed) == sum(torch.is_tensor(a) for a in args)
    _close(torch.autograd.grad(out, leaves, up), want)
    # operands changed in place
    first = args[0].detach().clone().requires_grad_()
    moved = first * 1
    out = KINDS[kind].apply(moved, *args[1:])
    moved.add_(1)
    with pytest.raises(RuntimeError, match="inplace"):
        (out if torch.is_tensor(out) else out[0]).sum().backward()
    # recomputed in the backward
    for reentrant in (True, False):
        got = checkpoint(lambda v: KINDS[kind].apply(v * 1, *args[1:]), first, use_reentrant=reentrant)
        got = got if isinstance(got, tuple) else (got,)
        _close(torch.autograd.grad(got, [first], up) if not reentrant else _backward(got, up, first), want[:1])
    with torch.autograd.detect_anomaly(check_nan=False):
        out, leaves = _record(kind, args)
        _close(torch.autograd.grad(out, leaves, up), want)


def _backward(out, up, leaf):
    leaf.grad = None
    torch.autograd.backward(out, up)
    return [leaf.grad]


@pytest.mark.parametrize("kind", KINDS)
def test_compiled_autograd(kind):
    from torch._dynamo import compiled_autograd
    args = _args(kind)
    out, leaves = _record(kind, args)
    up = _upstream(out)
    want = torch.autograd.grad(out, leaves, up, retain_graph=True)
    with compiled_autograd._enable(lambda graph: graph):
        _close(torch.autograd.grad(out, leaves, up), want)


def test_who_sees_the_call_has_a_python_node():
    args = _args("fused")
    from dfa3D import _lib

    def native():
        return _is_native(_record("fused", args)[0][0])
    assert native()
    with torch.autocast("cuda"):
        assert not native()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):
        assert not native()
    with _lib.launch_options(iters=2):
        assert not native()
    with torch.no_grad():
        assert KINDS["fused"].apply(*args)[0].grad_fn is None
    assert KINDS["fused"].apply(*args)[0].grad_fn is None                   # nothing that has a gradient
    with pytest.raises(RuntimeError):
        KINDS["fused"].apply(args[0].cpu(), *args[1:])


def test_on_streams_of_its_own():
    """The backward runs on the stream of its forward, whichever is current when it is asked for."""
    args = _args("fused")
    out, leaves = _record("fused", args)
    up = _upstream(out)
    want = torch.autograd.grad(out, leaves, up)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out, leaves = _record("fused", args)
    side.synchronize()
    got = torch.autograd.grad(out, leaves, up)
    side.synchronize()
    _close(got, want)
    with torch.autograd.set_multithreading_enabled(False):
        out, leaves = _record("fused", args)
        _close(torch.autograd.grad(out, leaves, up), want)
