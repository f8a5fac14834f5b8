"""The linear layers around the operator: ``nn.Linear`` with its products formed by this package's own kernels
(csrc/dfa3d_linear.hip) where they apply.  A cross-attention layer projects 10^5 rows (the pixels of six cameras, or
the queries re-batched per camera) with weights of 256 x 256: the gradient of such a weight is a product with a tiny
result and a very long inner dimension."""
import torch
import torch.nn.functional as F
from torch import nn
from torch.autograd import Function
from torch.nn.modules import module as _module

from .. import _lib

__all__ = ["Projection", "projections", "projection_plus"]

_PLAIN = (torch.Tensor, nn.Parameter)


def ordinary(*tensors, dtype=torch.float32):
    """Plain tensors of ``dtype`` on one GPU, outside autocast, functorch transforms, dispatch modes, forward-mode derivatives,
    tracing and compilation: what this package's kernels may stand in for torch operations on."""
    return (not torch.compiler.is_compiling() and not torch.jit.is_tracing() and not torch.is_autocast_enabled()
            and torch._C._len_torch_dispatch_stack() == 0
            and all(type(t) in _PLAIN and t.is_cuda and t.dtype == dtype and not t.is_neg()
                    and t.device == tensors[0].device for t in tensors)
            and torch._C._functorch.peek_interpreter_stack() is None
            and torch.autograd.forward_ad._current_level < 0)


def _widths_apply(O, K):
    """Where the kernel takes the gradient of an O x K weight: even widths of up to 2048 whose product is at most 2^20.  The
    library's product is slow where the result has few tiles, and has caught up at about 64 tiles of 128 x 128.  The rule also bounds the
    workspace, 512 to 1024 tiles of 64 KB (2048 x 2048 would take 134 MB, 16384 x 16384 8.6 GB).  Times as fast as the library's product and
    column sum, 4096 / 20000 / 100000 rows: 256 x 512 1.5 / 4.5 / 4.1, 256 x 2048 1.2 / 1.8 / 1.3, 512 x 1024 1.2 / 1.0 / 1.0, 1024 x 1024
    1.05 / 0.95 / 1.1; beyond, 1024 x 2048 0.89 / 0.87 / 0.87, 2048 x 2048 0.84 / 0.87 / 0.85, 64 x 4096 1.1 / 0.9 / 0.8.
    Fewer rows, library and kernels, us a call (on the device alone): 256 x 256 16 rows 26 / 13 (14 / 10), 128 42 / 13 (41 / 10), 1000
    235 / 16 (234 / 15), 2000 30 / 21 (28 / 21); 512 x 256 16 rows 26 / 13 (7 / 11), 128 26 / 13 (10 / 11), 1000 30 / 17 (20 / 16); 128 x 128
    16 rows 26 / 13 (8 / 9), 300 30 / 13 (28 / 10)."""
    return O % 2 == 0 and K % 2 == 0 and max(O, K) <= 2048 and O * K <= 2 ** 20


def _product(x, weight, bias, addend=None):
    """``F.linear`` (plus ``addend``) that nothing records, or None where the kernel does not form it (csrc/dfa3d_binding.cpp says where
    it does) or it is to be recorded."""
    # (the type first: a symbolic tracer's proxy has no truth value)
    if (type(x) not in _PLAIN or not x.is_cuda or torch.compiler.is_compiling()
            or torch.autograd.forward_ad._current_level >= 0):
        return None
    native = _lib.binding()
    if native is None:
        return None
    at = torch._C._cuda_getDevice()
    return native.linear(at, torch._C._cuda_getCurrentRawStream(at), x, weight, bias, addend)


def _sum_of_products(operands):
    """Sum of rows (..., O) times weight (O, K) over the flat tuple of them, or None as above."""
    if not operands[0].is_cuda:
        return None
    native = _lib.binding()
    if native is None:
        return None
    at = torch._C._cuda_getDevice()
    return native.linear_sum(at, torch._C._cuda_getCurrentRawStream(at), operands)


def _linear(x, weight, bias, library):
    """``F.linear``, by the kernel where nothing records it and it is not to be the library's (``library``)."""
    got = None if library else _product(x, weight, bias)
    return F.linear(x, weight, bias) if got is None else got


def _linear_plus(x, weight, bias, addend):
    """``F.linear(x, weight, bias) + addend``, by the kernel where it forms the product and ``addend`` is as the result."""
    got = _product(x, weight, bias, addend)
    return F.linear(x, weight, bias) + addend if got is None else got


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


def _several_weight_gradients(x, grads, want_bias):
    """``_weight_gradients`` of several layers on the same rows, in the launches of one."""
    N, K = x.shape
    lib = _lib.lib()
    sizes = [lib.dfa3d_linear_grad_workspace_bytes(N, g.shape[1], K) for g in grads]
    workspace = torch.empty(sum(sizes), dtype=torch.uint8, device=x.device)
    out = [(x.new_empty(g.shape[1], K), x.new_empty(g.shape[1]) if want else None) for g, want in zip(grads, want_bias)]
    sets = (_lib.LinearGradSet * len(grads))(*((_lib.ptr(g), _lib.ptr(w), _lib.ptr(b), g.shape[1]) for g, (w, b) in zip(grads, out)))
    with _lib.on_device(x.device):
        rc = lib.dfa3d_linear_grads(_lib.ptr(x), sets, len(grads), _lib.ptr(workspace), sum(sizes), N, K, _lib.stream_of(x))
    _lib.check(rc, "dfa3d_linear_grads")
    return out


def plain_gradient(grad):
    """A gradient that a kernel may read: a plain float32 tensor on the GPU, not recorded and not a batch of gradients (is_grads_batched)."""
    return (type(grad) in _PLAIN and not torch.is_grad_enabled() and grad.is_cuda and grad.dtype == torch.float32
            and torch._C._len_torch_dispatch_stack() == 0 and torch.autograd.forward_ad._current_level < 0 and not grad.is_neg()
            and not torch._C._functorch.is_batchedtensor(grad) and not torch._C._functorch.is_legacy_batchedtensor(grad))


def as_plain(saved, grad):
    """A saved tensor (whatever a hook made of it) that a kernel may read beside the gradient."""
    return type(saved) in _PLAIN and saved.dtype == grad.dtype and saved.device == grad.device and saved.is_contiguous() and not saved.is_neg()


class _ProjectionFunction(Function):
    """``F.linear(x, weight, bias)`` with a bias; differentiable any number of times (a backward that is itself recorded
    is made of torch operations)."""

    @staticmethod
    def forward(ctx, x, weight, bias, library_forward=False):
        # each operand only where the other one's gradient needs it, as F.linear keeps them: the other may be changed in place
        want_x, want_weight = ctx.needs_input_grad[:2]
        ctx.save_for_backward(x if want_weight else None, weight if want_x else None)
        return _linear(x, weight, bias, library_forward)

    @staticmethod
    def backward(ctx, grad):
        x, weight = ctx.saved_tensors
        want_x, want_weight, want_bias = ctx.needs_input_grad[:3]
        if plain_gradient(grad):
            grad = grad.contiguous()
        return (_input_gradient([grad], [weight]) if want_x else None, *_layer_gradients(x, grad, want_weight, want_bias), None)


class _ProjectionPlusFunction(Function):
    """``F.linear(x, weight, bias) + addend``, ``addend`` as the result."""

    @staticmethod
    def forward(ctx, x, weight, bias, addend):
        want_x, want_weight = ctx.needs_input_grad[:2]
        ctx.save_for_backward(x if want_weight else None, weight if want_x else None)
        return _linear_plus(x, weight, bias, addend)

    @staticmethod
    def backward(ctx, grad):
        return *_ProjectionFunction.backward(ctx, grad)[:3], grad if ctx.needs_input_grad[3] else None


def _input_gradient(grads, weights):
    """Gradient of the rows that several layers share, from the gradients of what they gave."""
    if all(plain_gradient(g) for g in grads):
        got = _sum_of_products(tuple(t for pair in zip(grads, weights) for t in pair))
        if got is not None:
            return got
    total = grads[0].matmul(weights[0])
    for g, w in zip(grads[1:], weights[1:]):
        total = total + g.matmul(w)
    return total


def _layer_gradients(x, grad, want_weight, want_bias):
    """Gradients of a layer's weight and bias from its rows x and the gradient of its result."""
    grad_rows = grad.reshape(-1, grad.shape[-1])
    if not want_weight:
        return None, grad_rows.sum(0) if want_bias else None
    rows = x.reshape(-1, x.shape[-1]).contiguous()
    if not (plain_gradient(grad) and as_plain(rows, grad)):
        return grad_rows.t().mm(rows), grad_rows.sum(0) if want_bias else None
    return _weight_gradients(rows, grad_rows.contiguous(), want_bias)


class _SharedRowsFunction(Function):
    """``F.linear(x, weight, bias)`` of several layers (weight, bias, weight, bias, ...) on the same rows; ``library``
    says whose forward is the library's.  The gradient of the rows is formed in one kernel instead of one product per
    layer and the sums of their results."""

    @staticmethod
    def forward(ctx, library, x, *params):
        weights, biases = params[::2], params[1::2]
        ctx.set_materialize_grads(False)
        want_x, *wanted = ctx.needs_input_grad[1:]
        ctx.save_for_backward(x if any(wanted[::2]) else None, *(w if want_x else None for w in weights))
        return tuple(_linear(x, w, b, lib) for w, b, lib in zip(weights, biases, library))

    @staticmethod
    def backward(ctx, *grads):
        x, *weights = ctx.saved_tensors
        want_x, *wanted = ctx.needs_input_grad[1:]
        grads = [g.contiguous() if g is not None and plain_gradient(g) else g for g in grads]
        there = [i for i, g in enumerate(grads) if g is not None]
        grad_x = _input_gradient([grads[i] for i in there], [weights[i] for i in there]) if want_x and there else None
        out = [None] * (2 * len(grads))
        together = [i for i in there if wanted[2 * i]]         # (the layers whose weight's gradient is wanted)
        rows = x.reshape(-1, x.shape[-1]).contiguous() if len(together) > 1 else None
        if rows is not None and all(plain_gradient(grads[i]) and as_plain(rows, grads[i]) for i in together):
            formed = _several_weight_gradients(rows, [grads[i].reshape(-1, grads[i].shape[-1]) for i in together],
                                               [wanted[2 * i + 1] for i in together])
            for i, pair in zip(together, formed):
                out[2 * i:2 * i + 2] = pair
        else:
            together = ()
        for i in there:
            if i not in together:
                out[2 * i:2 * i + 2] = _layer_gradients(x, grads[i], *wanted[2 * i:2 * i + 2])
        return (None, grad_x, *out)


def _applies(x, *layers):
    """Float32 rows on the GPU in ordinary reverse-mode training, for layers that all have a bias."""
    return (not torch.compiler.is_compiling() and torch.is_grad_enabled() and x.dim() >= 2
            and 0 < x.numel() // max(x.shape[-1], 1) <= 2 ** 31
            and all(l.bias is not None and l.weight.requires_grad and _widths_apply(*l.weight.shape) for l in layers)
            and ordinary(x, *(t for l in layers for t in (l.weight, l.bias))))


class Projection(nn.Linear):
    """``nn.Linear``: same parameters, same results.

    ``library_forward``: the result is the library's to the bit.  For sampling offsets: the gradient of a sampling
    location jumps where the location passes from one pixel or depth bin to the next, so two products that round
    differently, neither of them further from the exact one, put some hundred of 15 million points on the other side,
    and gradients differ by 7e-4."""

    library_forward = False

    def __init__(self, in_features, out_features, bias=True, device=None, dtype=None, library_forward=False):
        super().__init__(in_features, out_features, bias, device, dtype)
        self.library_forward = library_forward

    def forward(self, input):
        if _applies(input, self):
            return _ProjectionFunction.apply(input, self.weight, self.bias, self.library_forward)
        return _linear(input, self.weight, self.bias, self.library_forward)


def no_hooks(layer):
    """Whether the module's call is its class's ``forward`` and nothing else."""
    return ("forward" not in layer.__dict__
            and not (layer._forward_hooks or layer._forward_pre_hooks or layer._backward_hooks or layer._backward_pre_hooks
                     or _module._global_forward_hooks or _module._global_forward_pre_hooks
                     or _module._global_backward_hooks or _module._global_backward_pre_hooks))


def _bare(layer):
    return type(layer) is Projection and no_hooks(layer)


def projection_plus(layer, x, addend):
    """``layer(x) + addend`` without a pass over the result for the sum: the layer of the small model, inference, 252 -> 246 us."""
    if _bare(layer) and not layer.library_forward and type(addend) in _PLAIN and addend.shape == (*x.shape[:-1], layer.out_features):
        if _applies(x, layer) and ordinary(x, addend):
            if addend.is_contiguous():
                return _ProjectionPlusFunction.apply(x, layer.weight, layer.bias, addend)
        elif (got := _product(x, layer.weight, layer.bias, addend)) is not None:
            return got
    return layer(x) + addend


def projections(x, layers):
    """``[layer(x) for layer in layers]``; where the layers are plain ``Projection``s, at most four, the gradient of
    ``x`` is formed in one kernel.  The layer of the base model, training: 3811 -> 3771 us."""
    if len(layers) <= _lib.MAX_LINEAR_SETS and all(_bare(l) for l in layers) and _applies(x, *layers):
        params = [t for l in layers for t in (l.weight, l.bias)]
        return list(_SharedRowsFunction.apply(tuple(l.library_forward for l in layers), x, *params))
    return [layer(x) for layer in layers]
