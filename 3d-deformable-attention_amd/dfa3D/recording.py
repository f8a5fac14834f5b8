"""Calls of an autograd Function that nothing records."""
import torch
from torch import _functorch
from torch.autograd.function import Function

from . import _lib

__all__ = ["OperatorFunction"]


class _Notes:
    """What a forward keeps for its backward, where there will be none."""

    needs_input_grad = ()

    def save_for_backward(self, *tensors):
        pass

    def set_materialize_grads(self, value):
        pass


class OperatorFunction(Function):
    """A Function whose ``apply`` is its ``forward`` where gradients are off: making a node and wrapping what comes back is 4 of
    the 12 us that a forward of 2 x 100 queries takes.  Tracing, compilation, functorch transforms, forward mode, and profilers and
    other observers, which see a call or refuse it, have the node made all the same, as do subclasses from elsewhere (and all calls where there is no
    binding module to say who sees them; asked one by one from here they are 0.2 us of 9).  A class says with ``own = True`` in its own body that its ``forward`` asks no more of its context than ``_Notes``
    has and returns none of its operands: ``Function`` hands out another tensor where a forward does, this the operand itself."""

    own = False

    @classmethod
    def apply(cls, *args, **kwargs):
        # gradients first: a training step's calls are not to pay for the other questions (1.5 us of 27 a forward, of which 0.5 is left)
        if (torch.is_grad_enabled() or torch.compiler.is_compiling() or kwargs or not cls.__dict__.get("own", False)
                or torch.autograd.forward_ad._current_level >= 0 or (native := _lib.binding()) is None or native.seen()):
            return super().apply(*args, **kwargs)
        return cls.forward(_Notes(), *_functorch.utils.unwrap_dead_wrappers(args))
