"""Native nodes where something else than plain tensors and the engine has a part in the backward."""
import pytest
import torch
from torch.utils._pytree import tree_map

from dfa3D import functional as f
from dfa3D.modules.ms_deform_attn_3d import _SamplingFunction
from dfa3D.modules.projection import Projection, projection_plus, projections
from test_gpu_native_nodes import KINDS, _args, _close, _is_native, _record, _upstream
from test_gpu_parity import _dev

pytestmark = pytest.mark.gpu


@pytest.fixture
def by_python(monkeypatch):
    """The kinds whose backward ran in Python."""
    kinds, run = [], f.backward_of
    monkeypatch.setattr(f, "backward_of", lambda kind, *rest: kinds.append(kind) or run(kind, *rest))
    return kinds


class _Seen(torch.Tensor):
    """A tensor whose operations go through Python, on memory of its own."""

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        plain = lambda o: o.as_subclass(torch.Tensor) if type(o) is _Seen else o
        with torch._C._DisableTorchDispatch():
            out = func(*map(plain, args), **{k: plain(v) for k, v in (kwargs or {}).items()})
        return torch.Tensor._make_subclass(_Seen, out) if func is torch.ops.aten.detach.default else out      # (what is unpacked is detached)


@pytest.mark.parametrize("kind", KINDS)
def test_saved_tensors_that_a_hook_makes_dispatch_to_python(kind, by_python):
    args = _args(kind)
    out, leaves = _record(kind, args)
    up = _upstream(out)
    want = torch.autograd.grad(out, leaves, up)
    assert not by_python
    made = lambda t: torch.Tensor._make_subclass(_Seen, t.detach()) if t.is_floating_point() else t
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, made):
        out, leaves = _record(kind, args)
    assert _is_native(out[0])
    _close([g.as_subclass(torch.Tensor) for g in torch.autograd.grad(out, leaves, up)], want)
    assert len(by_python) == 1


class _Held(torch.Tensor):
    """A tensor without memory of its own, whose operations go through Python to the one it holds."""

    @staticmethod
    def __new__(cls, t):
        made = torch.Tensor._make_wrapper_subclass(cls, t.shape, strides=t.stride(), dtype=t.dtype, device=t.device)
        made.held = t
        return made

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        held = lambda o: o.held if isinstance(o, _Held) else o
        out = func(*tree_map(held, args), **tree_map(held, kwargs or {}))
        return _Held(out) if func is torch.ops.aten.detach.default else out


@pytest.mark.parametrize("rows", [100, 5000])
def test_layers_whose_saved_tensors_are_held_elsewhere(rows):
    """Projections on the same rows, one with a residual, and the sampling locations: tensor operations, where a kernel would find no memory."""
    dev = _dev()
    g = torch.Generator(device=dev).manual_seed(rows)
    rand = lambda *s: torch.randn(*s, generator=g, device=dev)
    layers = [Projection(32, O).to(dev) for O in (16, 8)]
    x, residual = rand(2, rows, 32).requires_grad_(), rand(2, rows, 16)
    uv, dz, logits = (rand(*s).requires_grad_() for s in ((1, rows, 2, 1, 4, 2), (1, rows, 2, 1, 4, 1), (1, rows, 2, 1, 4)))
    table, ref = torch.tensor([[6, 9, 5]], device=dev), rand(1, rows, 2, 3)
    leaves = [x, uv, dz, logits] + [p for l in layers for p in l.parameters()]
    up = [rand(2, rows, 16), rand(2, rows, 8), rand(2, rows, 16), rand(1, rows, 2, 1, 4, 3), rand(1, rows, 2, 1, 4)]

    def outputs():
        return [*projections(x, layers), projection_plus(layers[0], x, residual), *_SamplingFunction.apply(uv, dz, logits, ref, table)]

    want = torch.autograd.grad(outputs(), leaves, up)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach(), _Held):
        out = outputs()
    for a, b in zip(torch.autograd.grad(out, leaves, up), want):
        assert type(a) is torch.Tensor
        assert (a - b).norm() <= 2e-6 * b.norm()               # sums in another order


@pytest.mark.parametrize("kind", KINDS)
def test_a_profiler_that_comes_for_the_backward_sees_it(kind, by_python):
    args = _args(kind)
    out, leaves = _record(kind, args)
    up = _upstream(out)
    want = torch.autograd.grad(out, leaves, up, retain_graph=True)
    assert _is_native(out[0]) and not by_python
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):
        got = torch.autograd.grad(out, leaves, up)
    _close(got, want)
    assert len(by_python) == 1


@pytest.mark.parametrize("kind", KINDS)
def test_what_a_node_shows(monkeypatch, kind):
    """The class's name, the tensors that are saved and the step, as a node made in Python has them."""
    args = _args(kind)
    args[-1] = 32
    shown = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(KINDS[kind], "kind", None)
        out, leaves = _record(kind, args)
        node = out[0].grad_fn
        assert _is_native(out[0]) == native and node.im2col_step == 32 and isinstance(node.saved_tensors, tuple)
        for t, a in zip(node.saved_tensors, args):
            assert torch.equal(t, a) and t.requires_grad == a.is_floating_point()
        shown.append((type(node).__name__, len(node.saved_tensors), tuple(node.needs_input_grad)[:len(args)], [n is None for n, _ in node.next_functions]))
        torch.autograd.grad(out, leaves, _upstream(out))
        with pytest.raises(RuntimeError, match="second time"):
            node.saved_tensors
    assert shown[0] == shown[1]
    monkeypatch.undo()
    hooked = torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda())
    with hooked:
        out, _ = _record(kind, args)
    assert _is_native(out[0]) and all(t.is_cuda and torch.equal(t, a) for t, a in zip(out[0].grad_fn.saved_tensors, args))
    first = [a.requires_grad_() if i == 0 else a for i, a in enumerate(_args(kind))]
    out = KINDS[kind].apply(*first)
    node = (out if torch.is_tensor(out) else out[0]).grad_fn
    assert node.needs_input_grad == (True,) + (False,) * (len(first) - 1)
