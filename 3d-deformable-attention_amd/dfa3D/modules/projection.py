"""The linear layers around the operator: ``nn.Linear`` with the weight and bias gradients formed by the library's own
kernel (csrc/dfa3d_linear.hip) where that applies.  A cross-attention layer projects 10^5 rows (the pixels of six cameras, or
the queries re-batched per camera) with weights of 256 x 256: the gradient of such a weight is a product with a tiny
result and a very long inner dimension."""
import torch
import torch.nn.functional as F
from torch import nn
from torch.autograd import Function

from .. import _lib

__all__ = ["Projection"]


def ordinary(*tensors):
    """Plain float32 tensors on one GPU, outside autocast, functorch transforms, forward-mode derivatives, tracing and
    compilation: what this package's kernels may stand in for torch operations on."""
    return (not torch.compiler.is_compiling() and not torch.jit.is_tracing() and not torch.is_autocast_enabled()
            and all(type(t) in (torch.Tensor, nn.Parameter) and t.is_cuda and t.dtype == torch.float32
                    and t.device == tensors[0].device for t in tensors)
            and torch._C._functorch.peek_interpreter_stack() is None
            and torch.autograd.forward_ad._current_level < 0)


# Fewer rows than this: the library product is as fast and there is one launch less.
_MIN_ROWS = 4096


def _widths_apply(O, K):
    """Where the kernel takes the gradient of an O x K weight: even widths of up to 2048 whose product is at most 2^20.  The
    library's product is slow where the result has few tiles, and has caught up at about 64 tiles of 128 x 128.  Times as
    fast as the library's product and column sum, 4096 / 20000 / 100000 rows: 256 x 512 1.5 / 4.5 / 4.1, 256 x 2048 1.2 /
    1.8 / 1.3, 512 x 1024 1.2 / 1.0 / 1.0, 1024 x 1024 1.05 / 0.95 / 1.1; beyond, 1024 x 2048 0.89 / 0.87 / 0.87, 2048 x 2048
    0.84 / 0.87 / 0.85, 64 x 4096 1.1 / 0.9 / 0.8.  The rule also bounds the workspace, 512 to 1024 tiles of 64 KB (2048 x
    2048 would take 134 MB, 16384 x 16384 8.6 GB)."""
    return O % 2 == 0 and K % 2 == 0 and max(O, K) <= 2048 and O * K <= 2 ** 20


def _weight_gradients(x, grad, want_bias):
    """grad_weight (O, K) and grad_bias (O) or None, of contiguous float32 rows x (N, K) and grad (N, O)."""
    N, K = x.shape
    O = grad.shape[1]
    grad_weight = torch.empty(O, K, dtype=torch.float32, device=x.device)
    grad_bias = torch.empty(O, dtype=torch.float32, device=x.device) if want_bias else None
    lib = _lib.lib()
    nbytes = lib.dfa3d_linear_grad_workspace_bytes(N, O, K)
    workspace = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    with _lib.on_device(x.device):
        rc = lib.dfa3d_linear_grad(_lib.ptr(x), _lib.ptr(grad), _lib.ptr(grad_weight), _lib.ptr(grad_bias),
                                   _lib.ptr(workspace), nbytes, N, O, K, _lib.stream_of(x))
    _lib.check(rc, "dfa3d_linear_grad")
    return grad_weight, grad_bias


def plain_gradient(grad):
    """A gradient that a kernel may read: float32 on the GPU, not recorded and not a batch of gradients (is_grads_batched)."""
    return (not torch.is_grad_enabled() and grad.is_cuda and grad.dtype == torch.float32
            and not torch._C._functorch.is_batchedtensor(grad) and not torch._C._functorch.is_legacy_batchedtensor(grad))


class _ProjectionFunction(Function):
    """``F.linear(x, weight, bias)`` with a bias; differentiable any number of times (a backward that is itself recorded
    is made of torch operations)."""

    @staticmethod
    def forward(ctx, x, weight, bias):
        # each operand only where the other one's gradient needs it, as F.linear keeps them: the other may be changed in place
        want_x, want_weight, _ = ctx.needs_input_grad
        ctx.save_for_backward(x if want_weight else None, weight if want_x else None)
        return F.linear(x, weight, bias)

    @staticmethod
    def backward(ctx, grad):
        x, weight = ctx.saved_tensors
        want_x, want_weight, want_bias = ctx.needs_input_grad
        grad_x = grad.matmul(weight) if want_x else None
        grad_rows = grad.reshape(-1, grad.shape[-1])
        if not want_weight:
            return grad_x, None, grad_rows.sum(0) if want_bias else None
        rows = x.reshape(-1, x.shape[-1])
        if not plain_gradient(grad):
            return grad_x, grad_rows.t().mm(rows), grad_rows.sum(0) if want_bias else None
        return (grad_x, *_weight_gradients(rows.contiguous(), grad_rows.contiguous(), want_bias))


def _applies(x, weight, bias):
    """Float32 rows on the GPU in ordinary reverse-mode training."""
    return (not torch.compiler.is_compiling() and bias is not None and torch.is_grad_enabled() and weight.requires_grad
            and x.dim() >= 2 and _widths_apply(*weight.shape)
            and _MIN_ROWS <= x.numel() // max(x.shape[-1], 1) <= 2 ** 31 and ordinary(x, weight, bias))


class Projection(nn.Linear):
    """``nn.Linear``: same parameters, same results."""

    def forward(self, input):
        if _applies(input, self.weight, self.bias):
            return _ProjectionFunction.apply(input, self.weight, self.bias)
        return F.linear(input, self.weight, self.bias)
