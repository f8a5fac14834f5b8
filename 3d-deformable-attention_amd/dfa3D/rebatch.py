"""Camera re-batching around the DFA3D operator: the BEV queries that project into each camera are copied into
a per-camera batch before the attention and the per-camera results are averaged back into the BEV slots
afterwards.  The reference does both in python loops over batch x cameras
(BEVFormer_DFA3D/projects/mmdet3d_plugin/bevformer/modules/spatial_cross_attention.py:716-722, 741-748);
here each direction is one HIP kernel (csrc/dfa3d_rebatch.hip), and each kernel is the other's backward."""
import torch
from torch.autograd.function import once_differentiable

from . import _lib
from .recording import OperatorFunction

__all__ = ["camera_hits", "camera_count", "camera_hits_counted", "camera_index", "rebatch_gather", "rebatch_queries", "rebatch_combine",
           "RebatchGatherFunction", "RebatchQueriesFunction", "RebatchCombineFunction"]


def camera_count(hit):
    """Starts counting the queries of each camera of ``hit`` (cams, Nq) and the copy of the counts to the host: hand the result
    to ``camera_index``, which then waits for these alone and not for what was launched in between.  None where the lists
    are not made by the kernels."""
    cams, Nq = hit.shape
    if not (hit.is_cuda and hit.dtype == torch.bool and hit.is_contiguous() and 0 < cams <= 65535 and 0 < Nq <= 2 ** 30):
        return None
    totals = torch.empty(cams, dtype=torch.int32, device=hit.device)
    with _lib.on_device(hit.device):
        rc = _lib.lib().dfa3d_camera_count(_lib.ptr(hit), _lib.ptr(totals), cams, Nq, _lib.stream_of(hit))
        _lib.check(rc, "dfa3d_camera_count")
        return _on_their_way(totals)


def _on_their_way(counts):
    """``counts`` (cams,) or (cams, parts) on the GPU, the same on the host, and the event after which the host has them."""
    on_host = torch.empty(counts.shape, dtype=torch.int32, device="cpu", pin_memory=True)      # (whatever the default device)
    on_host.copy_(counts, non_blocking=True)
    done = torch.cuda.Event()
    done.record()
    return counts, on_host, done


# Workgroups that count, 1024 queries each at a time, and up to how many queries of all batch elements they count as they mark the
# hits; with more of them, workgroups that mark alone are as many as there are queries for.
_PARTS, _COUNTED_QUERIES = 64, 2 ** 18


def camera_hits_counted(bev_mask):
    """``camera_hits(bev_mask)`` and ``camera_count`` of its first result, in one launch where both are the kernels' and queries are not many."""
    cams, bs, Nq, Z = bev_mask.shape
    if not (_hits_by_kernel(bev_mask) and cams <= 1024 and bs * Nq <= _COUNTED_QUERIES):
        hit, scale = camera_hits(bev_mask)
        return hit, scale, camera_count(hit)
    mask = bev_mask.contiguous()
    parts = min(-(-bs * Nq // 1024), _PARTS)
    hit = torch.empty(cams, Nq, dtype=torch.bool, device=mask.device)
    scale = torch.empty(bs, Nq, dtype=torch.float32, device=mask.device)
    counts = torch.empty(cams, parts, dtype=torch.int32, device=mask.device)
    with _lib.on_device(mask.device):
        rc = _lib.lib().dfa3d_camera_hits_counted(_lib.ptr(mask), _lib.ptr(hit), _lib.ptr(scale), _lib.ptr(counts), parts, cams, bs, Nq, Z,
                                                  _lib.stream_of(mask))
        _lib.check(rc, "dfa3d_camera_hits_counted")
        return hit, scale, _on_their_way(counts)


def camera_index(hit, counted=None):
    """``hit`` (cams, Nq) bool: query q projects into camera i.  Returns ``index`` (cams, max_len) int32, the
    queries of each camera in ascending order padded with -1, and its inverse ``pos`` (cams, Nq) int32
    (position of q in camera i's list, or -1).  ``max_len`` depends on the data, so this synchronises with the
    device once, like the reference's ``nonzero`` calls (spatial_cross_attention.py:704-707).  ``counted``: what
    ``camera_count`` returned for this very ``hit``."""
    hit = hit.bool().contiguous()
    if counted is None:
        counted = camera_count(hit)
    if counted is not None:
        return _camera_index_on_gpu(hit, *counted)
    rank = hit.cumsum(1, dtype=torch.int32) - 1                      # position among the camera's queries
    pos = torch.where(hit, rank, torch.full_like(rank, -1)).contiguous()
    max_len = int(hit.sum(1).max().item()) if hit.numel() else 0
    index = torch.full((hit.shape[0], max(max_len, 1)), -1, dtype=torch.int32, device=hit.device)
    cam, q = hit.nonzero(as_tuple=True)
    index[cam, rank[cam, q].long()] = q.to(torch.int32)
    return index, pos, max_len


def _camera_index_on_gpu(hit, _, on_host, done):
    cams, Nq = hit.shape
    dev, lib = hit.device, _lib.lib()
    pos = torch.empty(cams, Nq, dtype=torch.int32, device=dev)
    with _lib.on_device(dev):
        done.synchronize()                                          # waits for the device
        max_len = max(map(sum, on_host.view(cams, -1).tolist()))
        index = torch.empty(cams, max(max_len, 1), dtype=torch.int32, device=dev)
        _lib.check(lib.dfa3d_camera_index(_lib.ptr(hit), None, _lib.ptr(index), _lib.ptr(pos), cams, Nq,
                                          max(max_len, 1), _lib.stream_of(hit)), "dfa3d_camera_index")
    return index, pos, max_len


def _hits_by_kernel(bev_mask):
    cams, _, Nq, _ = bev_mask.shape
    return (bev_mask.is_cuda and bev_mask.dtype == torch.bool and bev_mask.numel() and cams <= 65535 and Nq <= 2 ** 30
            and torch.get_default_dtype() == torch.float32)            # what the kernel writes


def camera_hits(bev_mask):
    """``bev_mask`` (cams, bs, Nq, Z): ``hit`` (cams, Nq) bool, the queries of the first batch element with any anchor in a
    camera, and ``scale`` (bs, Nq) of the default dtype, one over the number of cameras with any anchor of a query (at
    least 1)."""
    cams, bs, Nq, Z = bev_mask.shape
    if _hits_by_kernel(bev_mask):
        mask = bev_mask.contiguous()
        hit = torch.empty(cams, Nq, dtype=torch.bool, device=mask.device)
        scale = torch.empty(bs, Nq, dtype=torch.float32, device=mask.device)
        with _lib.on_device(mask.device):
            rc = _lib.lib().dfa3d_camera_hits(_lib.ptr(mask), _lib.ptr(hit), _lib.ptr(scale), cams, bs, Nq, Z,
                                              _lib.stream_of(mask))
        _lib.check(rc, "dfa3d_camera_hits")
        return hit, scale
    seen = bev_mask.sum(-1) > 0                                              # (cams, bs, Nq)
    return seen[:, 0], 1.0 / torch.clamp(seen.permute(1, 2, 0).sum(-1), min=1.0)


def _check(t, name, dtype=None):
    if not t.is_cuda:
        raise RuntimeError(f"{name} must be a CUDA tensor")
    if not t.is_contiguous():
        raise RuntimeError(f"{name} tensor has to be contiguous")
    if dtype is not None and t.dtype != dtype:
        raise RuntimeError(f"{name} has dtype {t.dtype}, expected {dtype}")


def rebatch_gather(src, index, scale=None, per_camera=False, pad=0.0):
    """``src`` (bs, Nq, E), or (cams, bs, Nq, E) with ``per_camera`` -> (bs, cams, max_len, E):
    row [j, i, k] = scale[j, q] * src[(i,) j, q] with q = index[i, k], ``pad`` where index is -1."""
    _check(src, "src")
    _check(index, "index", torch.int32)
    cams, max_len = index.shape
    if per_camera:
        if src.dim() != 4 or src.shape[0] != cams:
            raise RuntimeError(f"src must be (cams, bs, Nq, E), got {tuple(src.shape)}")
        _, bs, Nq, E = src.shape
        cam_stride, batch_stride = bs * Nq * E, Nq * E
    else:
        if src.dim() != 3:
            raise RuntimeError(f"src must be (bs, Nq, E), got {tuple(src.shape)}")
        bs, Nq, E = src.shape
        cam_stride, batch_stride = 0, Nq * E
    if scale is not None:
        _check(scale, "scale", src.dtype)
        if tuple(scale.shape) != (bs, Nq):
            raise RuntimeError(f"scale must be (bs, Nq), got {tuple(scale.shape)}")
    dst = torch.empty(bs, cams, max_len, E, dtype=src.dtype, device=src.device)
    if dst.numel() == 0:
        return dst
    with _lib.on_device(src.device):
        rc = _lib.lib().dfa3d_rebatch_gather_padded(_lib.ptr(src), cam_stride, batch_stride, _lib.ptr(index), _lib.ptr(scale),
                                                    _lib.ptr(dst), bs, cams, max_len, Nq, E, _lib.dtype_code(src), pad,
                                                    _lib.stream_of(src))
    _lib.check(rc, "dfa3d_rebatch_gather")
    return dst


def rebatch_queries(src, plus, ref, index, ref_pad=0.0):
    """``src`` and ``plus`` (bs, Nq, E; or None), ``ref`` (cams, bs, Nq, R) -> (bs, cams, max_len, E) and (bs, cams, max_len, R): what
    ``rebatch_gather(src + plus, index)`` and ``rebatch_gather(ref, index, per_camera=True, pad=ref_pad)`` give."""
    for t, name, dtype in ((src, "src", None), (plus, "plus", src.dtype), (ref, "ref", src.dtype), (index, "index", torch.int32)):
        if t is not None:
            _check(t, name, dtype)
    cams, max_len = index.shape
    if src.dim() != 3 or ref.dim() != 4 or tuple(ref.shape[:3]) != (cams, *src.shape[:2]) or (plus is not None and plus.shape != src.shape):
        raise RuntimeError(f"src and plus must be (bs, Nq, E) and ref (cams, bs, Nq, R), got {tuple(src.shape)}, "
                           f"{None if plus is None else tuple(plus.shape)}, {tuple(ref.shape)}")
    bs, Nq, E = src.shape
    R = ref.shape[3]
    dst, ref_dst = src.new_empty(bs, cams, max_len, E), src.new_empty(bs, cams, max_len, R)
    if dst.numel() == 0 or ref_dst.numel() == 0:
        return rebatch_gather(src if plus is None else src + plus, index), rebatch_gather(ref, index, per_camera=True, pad=ref_pad)
    with _lib.on_device(src.device):
        rc = _lib.lib().dfa3d_rebatch_queries(_lib.ptr(src), _lib.ptr(plus), _lib.ptr(ref), _lib.ptr(index), _lib.ptr(dst), _lib.ptr(ref_dst),
                                              bs, cams, max_len, Nq, E, R, _lib.dtype_code(src), ref_pad, _lib.stream_of(src))
    _lib.check(rc, "dfa3d_rebatch_queries")
    return dst, ref_dst


def rebatch_combine(src, pos, scale=None):
    """``src`` (bs, cams, max_len, E) -> (bs, Nq, E): row [j, q] = scale[j, q] * sum over the cameras i that see q
    of src[j, i, pos[i, q]]."""
    _check(src, "src")
    _check(pos, "pos", torch.int32)
    if src.dim() != 4 or pos.dim() != 2 or src.shape[1] != pos.shape[0]:
        raise RuntimeError(f"src must be (bs, cams, max_len, E) and pos (cams, Nq), got {tuple(src.shape)}, {tuple(pos.shape)}")
    bs, cams, max_len, E = src.shape
    Nq = pos.shape[1]
    if scale is not None:
        _check(scale, "scale", src.dtype)
        if tuple(scale.shape) != (bs, Nq):
            raise RuntimeError(f"scale must be (bs, Nq), got {tuple(scale.shape)}")
    dst = torch.empty(bs, Nq, E, dtype=src.dtype, device=src.device)
    if dst.numel() == 0:
        return dst
    if src.numel() == 0:
        return dst.zero_()
    with _lib.on_device(src.device):
        rc = _lib.lib().dfa3d_rebatch_combine(_lib.ptr(src), _lib.ptr(pos), _lib.ptr(scale), _lib.ptr(dst), bs, cams,
                                              max_len, Nq, E, _lib.dtype_code(src), _lib.stream_of(src))
    _lib.check(rc, "dfa3d_rebatch_combine")
    return dst


class RebatchGatherFunction(OperatorFunction):
    """``apply(src (bs, Nq, E), index, pos) -> (bs, cams, max_len, E)``; differentiable in ``src``."""

    own = True

    @staticmethod
    def forward(ctx, src, index, pos):
        ctx.save_for_backward(pos)
        return rebatch_gather(src.contiguous(), index)

    @staticmethod
    @once_differentiable
    def backward(ctx, grad):
        pos, = ctx.saved_tensors
        return rebatch_combine(grad.contiguous(), pos), None, None


class RebatchQueriesFunction(OperatorFunction):
    """``apply(src, plus or None, ref, index, pos, ref_pad)``: ``rebatch_queries``, differentiable in ``src`` and ``plus``."""

    own = True

    @staticmethod
    def forward(ctx, src, plus, ref, index, pos, ref_pad):
        ctx.save_for_backward(pos)
        ctx.set_materialize_grads(False)
        queries, refs = rebatch_queries(src.contiguous(), plus, ref, index, ref_pad)
        ctx.mark_non_differentiable(refs)
        return queries, refs

    @staticmethod
    @once_differentiable
    def backward(ctx, grad, _):
        if grad is None:
            return (None,) * 6
        pos, = ctx.saved_tensors
        grad = rebatch_combine(grad.contiguous(), pos)
        return tuple(grad if want else None for want in ctx.needs_input_grad[:2]) + (None,) * 4


class RebatchCombineFunction(OperatorFunction):
    """``apply(src (bs, cams, max_len, E), index, pos, scale (bs, Nq) or None) -> (bs, Nq, E)``; differentiable in
    ``src`` (``scale`` is a constant: the reciprocal camera count)."""

    own = True

    @staticmethod
    def forward(ctx, src, index, pos, scale):
        ctx.save_for_backward(index, scale)
        return rebatch_combine(src.contiguous(), pos, scale)

    @staticmethod
    @once_differentiable
    def backward(ctx, grad):
        index, scale = ctx.saved_tensors
        return rebatch_gather(grad.contiguous(), index, scale), None, None, None
