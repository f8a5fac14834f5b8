"""bfloat16 gradients where the cell-owned kernel's tiles are smaller than LDS allows: summed in float and rounded once, so
that their error is that of a single rounding; and with a workspace that has no room for the sums."""
import ctypes

import pytest
import torch

from test_gpu_parity import _dev

pytestmark = pytest.mark.gpu


def _operands(C, D, heads, dev):
    g = torch.Generator(device=dev).manual_seed(C + D)
    B, H, W, M, Q, P = 2, 41, 67, 8, 1500, 4
    value = torch.randn(B, H * W, M, C, generator=g, device=dev).bfloat16()
    dist = torch.randn(B, H * W, heads, D, generator=g, device=dev).softmax(-1).bfloat16()
    loc = torch.rand(B, Q, M, 1, P, 3, generator=g, device=dev)
    attn = torch.rand(B, Q, M, 1, P, generator=g, device=dev)
    go = torch.randn(B, Q, M * C, generator=g, device=dev).bfloat16()
    return (value, dist, torch.tensor([[H, W, D]], device=dev), torch.tensor([0], device=dev), loc, attn, go, None)


@pytest.mark.parametrize("clear", [False, True], ids=["zeroed", "anything"])
@pytest.mark.parametrize("heads", [8, 1], ids=["per-head", "shared"])
@pytest.mark.parametrize("C,D", [(4, 4), (16, 16), (28, 16), (40, 16), (64, 32)])
def test_gradients_are_rounded_once(C, D, heads, clear):
    from dfa3D import _ext
    args = _operands(C, D, heads, _dev())
    got = {}
    for dtype in (torch.float32, torch.bfloat16):
        gv, gd = (torch.full(t.shape, float("nan") if clear else 0.0, dtype=dtype, device=t.device) for t in args[:2])
        gl, ga = torch.empty_like(args[4]), torch.empty_like(args[5])
        _ext.dfa3d_fused_backward(*args, gv, gd, gl, ga, 64, clear=clear)
        got[dtype] = gv, gd
    for f, h in zip(got[torch.float32], got[torch.bfloat16]):
        once = (f.bfloat16().double() - f.double()).norm()
        # the float sums of two runs differ in their last bits, which moves a few elements across a rounding boundary
        assert (h.double() - f.double()).norm() <= 1.001 * once


def test_workspace_without_room_for_the_sums():
    """The C call takes the smaller workspace it took before, and adds in bfloat16."""
    from dfa3D import _ext, _lib
    dev, L = _dev(), _lib.lib()
    C, D = 64, 16
    value, dist, shapes, lsi, loc, attn, go, _ = _operands(C, D, 8, dev)
    B, S, M, _ = value.shape
    dims = (B, S, M, C, D, 1, loc.shape[1], loc.shape[4], M)
    full = L.dfa3d_fused_backward_workspace_bytes(*dims, _lib.DFA3D_BF16G, None)
    least = L.dfa3d_fused_backward_workspace_bytes(*dims, _lib.DFA3D_BF16, None)
    assert full >= least + 4 * (value.numel() + dist.numel())
    want = [torch.zeros(t.shape, device=dev) for t in (value, dist)]
    gl, ga = torch.empty_like(loc), torch.empty_like(attn)
    _ext.dfa3d_fused_backward(value, dist, shapes, lsi, loc, attn, go, None, *want, gl, ga, 64)
    gv, gd = torch.zeros_like(value), torch.zeros_like(dist)
    ws = torch.empty(least, dtype=torch.uint8, device=dev)
    p = _lib.ptr
    rc = L.dfa3d_fused_backward(p(value), p(dist), p(shapes), p(lsi), p(loc), p(attn), p(go), None, None, p(gv), p(gd), p(gl), p(ga),
                                p(ws), ctypes.c_size_t(least), *dims, _lib.DFA3D_BF16G, None, _lib.stream_of(value))
    assert rc == 0, L.dfa3d_last_error()
    for g, w in zip((gv, gd), want):
        assert ((g.double() - w.double()).norm() / w.double().norm()).item() < 2.0 ** -8      # up to four roundings of 2^-9
