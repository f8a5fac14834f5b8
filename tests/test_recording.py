"""Functions whose ``apply`` is their ``forward`` where nothing records: the same results, and a node all the same where somebody looks."""
import threading

import pytest
import torch
from torch.autograd import Function
from torch.autograd.function import once_differentiable

from dfa3D.recording import OperatorFunction


def _body():
    def forward(ctx, x, s):
        ctx.s = s
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(x)
        _body.seen.append(type(ctx).__name__)
        return x * ctx.s, x + 1

    def backward(ctx, g, h):
        return g * ctx.s, None
    return {"forward": staticmethod(forward), "backward": staticmethod(once_differentiable(backward))}


_body.seen = []
Plain = type("Plain", (Function,), _body())
Own = type("Own", (OperatorFunction,), dict(_body(), own=True))
Theirs = type("Theirs", (Own,), {})


def _took_the_short_way(call):
    _body.seen.clear()
    out = call()
    return out, _body.seen[-1] == "_Notes"


def test_without_gradients_the_forward_alone_runs():
    x = torch.randn(5, requires_grad=True)
    for mode in (torch.no_grad, torch.inference_mode):
        with mode():
            out, short = _took_the_short_way(lambda: Own.apply(x, 3))
            want = Plain.apply(x, 3)
        assert short
        for a, b in zip(out, want):
            assert torch.equal(a, b) and not a.requires_grad and a.grad_fn is None and a.is_inference() == b.is_inference()


def test_with_gradients_a_node_is_made():
    x = torch.randn(5, requires_grad=True)
    out, short = _took_the_short_way(lambda: Own.apply(x, 3))
    assert not short and torch.equal(torch.autograd.grad(out[0].sum(), x)[0], torch.full((5,), 3.0))
    out, short = _took_the_short_way(lambda: Own.apply(x.detach(), 3))
    assert not short and not out[0].requires_grad


def test_a_subclass_from_elsewhere_gets_a_context_of_torchs():
    with torch.no_grad():
        assert not _took_the_short_way(lambda: Theirs.apply(torch.ones(2), 3))[1]


def test_tracing_forward_mode_and_transforms_see_the_call():
    x = torch.randn(4)
    with torch.no_grad():
        traced = torch.jit.trace(lambda t: Own.apply(t, 3)[0], x, check_trace=False)
        assert any(n.kind() == "prim::PythonOp" for n in traced.graph.nodes())
        assert torch.equal(torch.compile(lambda t: Own.apply(t.sin(), 3)[0], backend="eager", fullgraph=True)(x), x.sin() * 3)
        for F in (Plain, Own):
            with pytest.raises(RuntimeError):
                torch.func.vmap(lambda t: F.apply(t, 3)[0])(x)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones(4))
        answers = []
        for F in (Plain, Own):
            with torch.no_grad():
                try:
                    answers.append(torch.autograd.forward_ad.unpack_dual(F.apply(dual, 3)[0]).tangent)
                except (RuntimeError, NotImplementedError) as e:
                    answers.append(type(e))
        assert answers[0] == answers[1]


def test_a_wrapper_left_over_from_a_transform_is_unwrapped():
    left = []
    torch.func.grad(lambda t: (left.append(t), t.sum())[1])(torch.ones(3))
    assert torch._C._functorch.is_functorch_wrapped_tensor(left[0])
    wrapped = []

    def forward(ctx, x):
        wrapped.append(torch._C._functorch.is_functorch_wrapped_tensor(x))
        return x * 3
    for base in (Function, OperatorFunction):
        F = type("F", (base,), {"own": True, "forward": staticmethod(forward)})
        with torch.no_grad():
            out = F.apply(left[0])
        assert torch.equal(out, torch.full((3,), 3.0)) and not torch._C._functorch.is_functorch_wrapped_tensor(out)
    assert wrapped == [False, False]


def test_export_sees_the_call():
    """Export without Dynamo runs ``apply`` itself, on tensors that hold nothing."""
    class M(torch.nn.Module):
        def forward(self, t):
            return Own.apply(t, 3)[0]
    x = torch.randn(4)
    with torch.no_grad():
        program, short = _took_the_short_way(lambda: torch.export.export(M(), (x,), strict=False))
        assert not short and torch.equal(program.module()(x), x * 3)


def test_a_profiler_sees_the_call(tmp_path):
    x = torch.randn(4)
    observer = torch.profiler.ExecutionTraceObserver().register_callback(str(tmp_path / "calls.json"))
    for mode in (torch.no_grad, torch.inference_mode):
        with mode():
            with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as seen:
                short = _took_the_short_way(lambda: Own.apply(x, 3))[1]
            assert not short and "Own" in [e.key for e in seen.key_averages()]
            observer.start()
            try:
                short = _took_the_short_way(lambda: Own.apply(x, 3))[1]
            finally:
                observer.stop()
            assert not short
            assert _took_the_short_way(lambda: Own.apply(x, 3))[1]
    observer.unregister_callback()
    assert '"Own"' in (tmp_path / "calls.json").read_text()


def test_without_a_binding_module_a_node_is_made(monkeypatch):
    from dfa3D import _lib
    _lib.lib()
    monkeypatch.setattr(_lib, "_binding", None)
    with torch.no_grad():
        out, short = _took_the_short_way(lambda: Own.apply(torch.ones(2), 3))
    assert not short and torch.equal(out[0], torch.full((2,), 3.0))


def test_with_gradients_nothing_else_is_asked(monkeypatch):
    """What a call that is recorded pays for the choice is the one question whether it is."""
    def asked():
        raise AssertionError("asked")
    monkeypatch.setattr(torch.compiler, "is_compiling", asked)
    x = torch.randn(4, requires_grad=True)
    assert Own.apply(x, 3)[0].requires_grad


def test_threads_do_not_share_a_context():
    results = [None] * 8

    def work(i):
        with torch.no_grad():
            results[i] = all(torch.equal(Own.apply(torch.full((3,), float(i)), i)[0], torch.full((3,), float(i * i))) for _ in range(200))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(results)
