"""The linear layers around the operator: ``nn.Linear`` with its products formed by this package's own kernels
(csrc/dfa3d_linear.hip) where they apply.  A cross-attention layer projects 10^5 rows (the pixels of six cameras, or
the queries re-batched per camera) with weights of 256 x 256: the gradient of such a weight is a product with a tiny
result and a very long inner dimension."""
import torch
import torch.nn.functional as F
from torch import nn
from torch.autograd import Function

from .. import _lib

__all__ = ["Projection"]


def ordinary(*tensors):
    """Plain float32 tensors on one GPU, outside autocast, functorch transforms, dispatch modes, forward-mode derivatives,
    tracing and compilation: what this package's kernels may stand in for torch operations on."""
    return (not torch.compiler.is_compiling() and not torch.jit.is_tracing() and not torch.is_autocast_enabled()
            and torch._C._len_torch_dispatch_stack() == 0
            and all(type(t) in (torch.Tensor, nn.Parameter) and t.is_cuda and t.dtype == torch.float32 and not t.is_neg()
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


def _product_applies(rows, width, depth):
    """Where the kernel forms a product of ``rows`` x ``width`` elements, sums of ``depth`` terms.  It reads four neighbours of a
    row at a time, and takes the library's place except where few rows meet a deep sum: library and kernel, us, 4096 rows
    of 256 by 256 19, 10; 256 by 64 19, 7; sums of 512 by 256 19, 22; of 2048 by 256 41, 51 to 89; of 1024 by 1024 72, 59; 20000 rows of 512 by
    512 98, 70; of 2048 by 256 165, 145; 100000 of 256 by 256 123, 93."""
    return width % 2 == 0 and depth % 4 == 0 and 0 < max(width, depth) <= 4096 and 0 < rows <= 2 ** 31 and \
        (depth <= 256 or rows * width >= 2 ** 22)


def _product(x, weight, bias, across):
    """x (..., K) times weight (O, K) transposed, or (``across``) weight (K, O), plus the bias; contiguous float32 operands."""
    O = weight.shape[1] if across else weight.shape[0]
    K = x.shape[-1]
    y = torch.empty(*x.shape[:-1], O, dtype=torch.float32, device=x.device)
    with _lib.on_device(x.device):
        rc = _lib.lib().dfa3d_linear(_lib.ptr(x), _lib.ptr(weight), _lib.ptr(bias), _lib.ptr(y), x.numel() // K, O, K, int(across),
                                     _lib.stream_of(x))
    _lib.check(rc, "dfa3d_linear")
    return y


def _linear(x, weight, bias):
    """``F.linear`` outside autograd."""
    if (x.is_cuda and x.is_contiguous() and weight.is_contiguous() and x.shape[-1:] == weight.shape[1:]
            and (bias is None or (bias.is_contiguous() and bias.shape == weight.shape[:1])) and _product_applies(x.numel() // max(x.shape[-1], 1), *weight.shape)):
        return _product(x, weight, bias, False)
    return F.linear(x, weight, bias)


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
            and torch._C._len_torch_dispatch_stack() == 0 and not grad.is_neg()
            and not torch._C._functorch.is_batchedtensor(grad) and not torch._C._functorch.is_legacy_batchedtensor(grad))


def _as_plain(saved, grad):
    """A saved tensor (whatever a hook made of it) that a kernel may read beside the gradient."""
    return saved.dtype == grad.dtype and saved.device == grad.device and saved.is_contiguous() and not saved.is_neg()


class _ProjectionFunction(Function):
    """``F.linear(x, weight, bias)`` with a bias; differentiable any number of times (a backward that is itself recorded
    is made of torch operations)."""

    @staticmethod
    def forward(ctx, x, weight, bias, library_forward=False):
        # each operand only where the other one's gradient needs it, as F.linear keeps them: the other may be changed in place
        want_x, want_weight = ctx.needs_input_grad[:2]
        ctx.save_for_backward(x if want_weight else None, weight if want_x else None)
        return F.linear(x, weight, bias) if library_forward else _linear(x, weight, bias)

    @staticmethod
    def backward(ctx, grad):
        x, weight = ctx.saved_tensors
        want_x, want_weight, want_bias = ctx.needs_input_grad[:3]
        plain = plain_gradient(grad)
        if plain:
            grad = grad.contiguous()
        grad_x = None
        if want_x:
            if plain and _as_plain(weight, grad) and _product_applies(grad.numel() // max(grad.shape[-1], 1), weight.shape[1], weight.shape[0]):
                grad_x = _product(grad, weight, None, True)
            else:
                grad_x = grad.matmul(weight)
        grad_rows = grad.reshape(-1, grad.shape[-1])
        if not want_weight:
            return grad_x, None, grad_rows.sum(0) if want_bias else None, None
        rows = x.reshape(-1, x.shape[-1]).contiguous()
        if not (plain and _as_plain(rows, grad)):
            return grad_x, grad_rows.t().mm(rows), grad_rows.sum(0) if want_bias else None, None
        return (grad_x, *_weight_gradients(rows, grad_rows, want_bias), None)


def _applies(x, weight, bias):
    """Float32 rows on the GPU in ordinary reverse-mode training."""
    return (not torch.compiler.is_compiling() and bias is not None and torch.is_grad_enabled() and weight.requires_grad
            and x.dim() >= 2 and _widths_apply(*weight.shape)
            and _MIN_ROWS <= x.numel() // max(x.shape[-1], 1) <= 2 ** 31 and ordinary(x, weight, bias))


def _no_gradient(x, weight, bias):
    """Float32 rows on the GPU that nothing records."""
    operands = (x, weight) if bias is None else (x, weight, bias)
    return (not torch.compiler.is_compiling() and x.is_cuda and not (torch.is_grad_enabled() and any(t.requires_grad for t in operands))
            and x.dim() >= 2 and ordinary(*operands))


class Projection(nn.Linear):
    """``nn.Linear``: same parameters, same results.

    ``library_forward``: in training the result is the library's to the bit.  For sampling offsets: the gradient of a sampling
    location jumps where the location passes from one pixel or depth bin to the next, so two products that round differently, neither
    of them further from the exact one, put some hundred of 15 million points on the other side, and gradients differ by 7e-4."""

    library_forward = False

    def __init__(self, in_features, out_features, bias=True, device=None, dtype=None, library_forward=False):
        super().__init__(in_features, out_features, bias, device, dtype)
        self.library_forward = library_forward

    def forward(self, input):
        if _applies(input, self.weight, self.bias):
            return _ProjectionFunction.apply(input, self.weight, self.bias, self.library_forward)
        if _no_gradient(input, self.weight, self.bias):
            return _linear(input, self.weight, self.bias)
        return F.linear(input, self.weight, self.bias)
