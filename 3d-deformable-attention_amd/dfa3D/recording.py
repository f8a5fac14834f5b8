"""Calls of an autograd Function without the interpreter's share: those that nothing records, and those whose node is native."""
import torch
from torch import _functorch
from torch.autograd.function import Function

from . import _ext, _lib

__all__ = ["OperatorFunction", "SCORE", "STAGE2", "PLAIN", "FUSED", "WEIGHT_UPDATE"]

SCORE, STAGE2, PLAIN, FUSED, WEIGHT_UPDATE = range(5)        # what the binding module calls and records as a whole


class _Notes:
    """What a forward keeps for its backward, where there will be none."""

    needs_input_grad = ()

    def save_for_backward(self, *tensors):
        pass

    def set_materialize_grads(self, value):
        pass

    def mark_non_differentiable(self, *results):
        pass


class OperatorFunction(Function):
    """A Function whose ``apply`` is its ``forward`` where gradients are off, and one call of the binding module, node and all, where that
    knows the call (``kind``) and takes its operands: making a node in Python and wrapping what comes back is 4 of the 12 us that a forward
    of 2 x 100 queries takes, and its backward holds the interpreter on the engine's thread.  Tracing, compilation, functorch transforms,
    forward mode, and profilers and other observers, which see a call or refuse it, have the Python node made all the same, as do autocast,
    launch options, subclasses from elsewhere (and all calls where there is no binding module to say who sees them; asked one by one from
    here they are 0.2 us of 9).  A class says with ``own = True`` in its own body that its ``forward`` asks no more of its context than
    ``_Notes`` has and returns none of its operands: ``Function`` hands out another tensor where a forward does, this the operand itself.
    A native node saves the operands as ``save_for_backward`` does and shows them, the step and the class's name as a node in Python does;
    where its backward is not one call of the library (a gradient that is recorded itself, operands that saved-tensor hooks have made into
    something else, an observer that has come since) it runs the class's own ``backward``."""

    own = False
    kind = None          # in a class's own body: the binding module knows the call as a whole

    @classmethod
    def apply(cls, *args, **kwargs):
        recorded = torch.is_grad_enabled()
        # (a class whose calls the binding module does not know asks no more where gradients are on)
        if ((recorded and cls.kind is None) or torch.compiler.is_compiling() or kwargs or not cls.__dict__.get("own", False)
                or torch.autograd.forward_ad._current_level >= 0 or (native := _lib.binding()) is None or native.seen()):
            return super().apply(*args, **kwargs)
        kind = cls.__dict__.get("kind")
        if kind is not None and args and isinstance(args[0], torch.Tensor):
            here = _ext._here(args[0])
            if here is not None and here[0] is native:
                got = native.call(here[1], here[2], kind, args)
                if got is not None:
                    return got
        if recorded:
            return super().apply(*args)
        return cls.forward(_Notes(), *_functorch.utils.unwrap_dead_wrappers(args))
