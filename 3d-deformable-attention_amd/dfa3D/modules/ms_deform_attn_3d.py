"""The attention module that calls the DFA3D operator in DFA3D-BEVFormer's spatial cross-attention,
without mmcv: same constructor arguments, parameter names (so the reference's checkpoints load with
``load_state_dict``), forward signature and results as ``MSDeformableAttention3D_DFA3D``
(BEVFormer_DFA3D/projects/mmdet3d_plugin/bevformer/modules/spatial_cross_attention.py:409-589, whose
constructor and value / offset / weight layers come from ``MSDeformableAttention3D``, :186-279).

Differences in how the same numbers are produced:
  * the depth distribution goes to the operator as (bs, keys, 1, D); the reference repeats it once per
    head (:496-497);
  * ``weight_update`` (:579) comes out of the operator's kernel; the (bs, Q, heads, L, P, 4) depth-score
    tensor is not materialised unless ``return_depth_score=True`` is passed to ``forward``.
"""
import math
import warnings

import torch
from torch import nn

from ..functional import (MultiScale3DDeformableAttnFunction_fp32,
                          MultiScale3DDeformableAttnWeightUpdateFunction_fp32)
from .. import _lib
from ..recording import OperatorFunction
from .projection import Projection, as_plain, ordinary, plain_gradient, projections

__all__ = ["MSDeformableAttention3D_DFA3D"]


def _readable(shapes3, grad):
    """Whether a kernel may read the saved level table (whatever a hook made of it) beside the gradient."""
    return type(shapes3) is torch.Tensor and shapes3.device == grad.device and shapes3.dtype == torch.int64 and shapes3.is_contiguous()


class _LocationsFunction(OperatorFunction):
    """uv (bs, Q, M, L, P, 2), dz (bs, Q, M, L, P, 1), reference points (bs, Q, Z, 3) and shapes (L, 3) to sampling locations
    in one kernel; differentiable in uv and dz, any number of times."""

    own = True

    @staticmethod
    def forward(ctx, uv, dz, reference_points, shapes3):
        ctx.save_for_backward(shapes3)
        bs, Q, M, L, P, _ = uv.shape
        loc = torch.empty(bs, Q, M, L, P, 3, dtype=torch.float32, device=uv.device)
        if loc.numel():
            with _lib.on_device(uv.device):
                rc = _lib.lib().dfa3d_locations(_lib.ptr(uv), _lib.ptr(dz), _lib.ptr(reference_points), _lib.ptr(shapes3),
                                                _lib.ptr(loc), bs * Q, M, L, P, reference_points.shape[2], _lib.stream_of(uv))
            _lib.check(rc, "dfa3d_locations")
        return loc

    @staticmethod
    def backward(ctx, grad):
        shapes3, = ctx.saved_tensors
        if not plain_gradient(grad) or not _readable(shapes3, grad) or grad.numel() == 0:
            scaled = grad / shapes3[:, [1, 0, 2]].to(grad.device, grad.dtype)[None, None, None, :, None, :]
            return scaled[..., :2], scaled[..., 2:], None, None
        grad = grad.contiguous()
        bs, Q, M, L, P, _ = grad.shape
        grad_uv, grad_dz = grad.new_empty(bs, Q, M, L, P, 2), grad.new_empty(bs, Q, M, L, P, 1)
        with _lib.on_device(grad.device):
            rc = _lib.lib().dfa3d_locations_grad(_lib.ptr(grad), _lib.ptr(shapes3), _lib.ptr(grad_uv), _lib.ptr(grad_dz), bs * Q,
                                                 M, L, P, _lib.stream_of(grad))
        _lib.check(rc, "dfa3d_locations_grad")
        return grad_uv, grad_dz, None, None


class _SamplingFunction(OperatorFunction):
    """As ``_LocationsFunction``, and logits (bs, Q, M, L, P) to their softmax over a head's points:
    ``apply(uv, dz, logits, reference_points, shapes3)``."""

    own = True

    @staticmethod
    def forward(ctx, uv, dz, logits, reference_points, shapes3):
        bs, Q, M, L, P = logits.shape
        loc, attn = logits.new_empty(bs, Q, M, L, P, 3), logits.new_empty(bs, Q, M, L, P)
        if attn.numel():
            with _lib.on_device(uv.device):
                rc = _lib.lib().dfa3d_sampling(_lib.ptr(uv), _lib.ptr(dz), _lib.ptr(logits), _lib.ptr(reference_points), _lib.ptr(shapes3),
                                               _lib.ptr(loc), _lib.ptr(attn), bs * Q, M, L, P, reference_points.shape[2], _lib.stream_of(uv))
            _lib.check(rc, "dfa3d_sampling")
        ctx.save_for_backward(shapes3, attn)
        return loc, attn

    @staticmethod
    def backward(ctx, grad_loc, grad_attn):
        shapes3, attn = ctx.saved_tensors
        if (not (plain_gradient(grad_loc) and plain_gradient(grad_attn) and as_plain(attn, grad_attn) and _readable(shapes3, attn))
                or attn.numel() == 0):
            scaled = grad_loc / shapes3[:, [1, 0, 2]].to(grad_loc.device, grad_loc.dtype)[None, None, None, :, None, :]
            weighted = grad_attn * attn
            return scaled[..., :2], scaled[..., 2:], weighted - attn * weighted.sum((-1, -2), keepdim=True), None, None
        grad_loc, grad_attn = grad_loc.contiguous(), grad_attn.contiguous()
        bs, Q, M, L, P = attn.shape
        grad_uv, grad_dz, grad_logits = attn.new_empty(bs, Q, M, L, P, 2), attn.new_empty(bs, Q, M, L, P, 1), attn.new_empty(attn.shape)
        with _lib.on_device(attn.device):
            rc = _lib.lib().dfa3d_sampling_grad(_lib.ptr(grad_loc), _lib.ptr(grad_attn), _lib.ptr(attn), _lib.ptr(shapes3), _lib.ptr(grad_uv),
                                                _lib.ptr(grad_dz), _lib.ptr(grad_logits), bs * Q, M, L, P, _lib.stream_of(attn))
        _lib.check(rc, "dfa3d_sampling_grad")
        return grad_uv, grad_dz, grad_logits, None, None


class MSDeformableAttention3D_DFA3D(nn.Module):
    """3D deformable attention over multi-scale image features with per-pixel depth distributions.

    Args (spatial_cross_attention.py:411, :212-221): embed_dims, num_heads, num_levels, num_points (sampling
    points per level and head, over all Z anchors), im2col_step, dropout (unused by the reference's forward as
    well), batch_first, norm_cfg, init_cfg (accepted, unused).
    """

    def __init__(self, embed_dims=256, num_heads=8, num_levels=4, num_points=8, im2col_step=64, dropout=0.1,
                 batch_first=True, norm_cfg=None, init_cfg=None):
        super().__init__()
        if embed_dims % num_heads != 0:
            raise ValueError(f"embed_dims must be divisible by num_heads, but got {embed_dims} and {num_heads}")
        dim_per_head = embed_dims // num_heads
        if dim_per_head & (dim_per_head - 1):
            warnings.warn("a power-of-two dimension per attention head lets every lane of a wavefront carry channels")
        self.norm_cfg = norm_cfg
        self.batch_first = batch_first
        self.output_proj = None
        self.fp16_enabled = False
        self.im2col_step = im2col_step
        self.embed_dims = embed_dims
        self.num_levels = num_levels
        self.num_heads = num_heads
        self.num_points = num_points
        self.sampling_offsets = Projection(embed_dims, num_heads * num_levels * num_points * 2, library_forward=True)
        self.attention_weights = Projection(embed_dims, num_heads * num_levels * num_points)
        self.value_proj = Projection(embed_dims, embed_dims)
        self.sampling_offsets_depth = Projection(embed_dims, num_heads * num_levels * num_points, library_forward=True)
        self.init_weights()
        self.init_smpl_off_weights()

    def init_weights(self):
        """Zero offset / weight matrices, offset biases on a ring of directions scaled by the point index,
        Xavier-uniform value projection (spatial_cross_attention.py:261-279)."""
        M, L, P = self.num_heads, self.num_levels, self.num_points
        with torch.no_grad():
            self.sampling_offsets.weight.zero_()
            thetas = torch.arange(M, dtype=torch.float32) * (2.0 * math.pi / M)
            ring = torch.stack([thetas.cos(), thetas.sin()], -1)
            ring = ring / ring.abs().max(-1, keepdim=True)[0]
            scale = torch.arange(1, P + 1, dtype=torch.float32).view(1, 1, P, 1)
            self.sampling_offsets.bias.copy_((ring.view(M, 1, 1, 2) * scale).expand(M, L, P, 2).reshape(-1))
            self.attention_weights.weight.zero_()
            self.attention_weights.bias.zero_()
            nn.init.xavier_uniform_(self.value_proj.weight)
            self.value_proj.bias.zero_()

    def init_smpl_off_weights(self):
        """Depth offsets: zero matrix, bias (cos + sin) / 2 of the head's direction times the point index
        (spatial_cross_attention.py:416-427)."""
        M, L, P = self.num_heads, self.num_levels, self.num_points
        with torch.no_grad():
            self.sampling_offsets_depth.weight.zero_()
            thetas = torch.arange(M, dtype=torch.float32) * (2.0 * math.pi / M)
            base = ((thetas.cos() + thetas.sin()) / 2).view(M, 1, 1)
            scale = torch.arange(1, P + 1, dtype=torch.float32).view(1, 1, P)
            self.sampling_offsets_depth.bias.copy_((base * scale).expand(M, L, P).reshape(-1))

    @staticmethod
    def get_spatial_shape_3D(spatial_shape, depth_dim):
        """(L, 2) -> (L, 3) with the number of depth bins as third extent (spatial_cross_attention.py:584-587)."""
        # one launch for two: a pass of the small model's layer has 18 others, most of them shorter than the host takes to make them
        # (for a number that the call takes as it is: numpy's, tensors, floats and what does not fit an int are torch's)
        if (type(depth_dim) is int and abs(depth_dim) < 2 ** 31 and spatial_shape.dim() == 2 and spatial_shape.shape[1] == 2
                and len(spatial_shape) and ordinary(spatial_shape, dtype=torch.int64) and spatial_shape.is_contiguous()):
            table = spatial_shape.new_empty(len(spatial_shape), 3)
            with _lib.on_device(table.device):
                rc = _lib.lib().dfa3d_level_table(_lib.ptr(spatial_shape), _lib.ptr(table), len(table), depth_dim, _lib.stream_of(table))
            _lib.check(rc, "dfa3d_level_table")
            return table
        depth = spatial_shape.new_full((*spatial_shape.shape[:-1], 1), depth_dim)
        return torch.cat([spatial_shape, depth], dim=-1).contiguous()

    def pack_dist(self, value_dpt_dist, spatial_shapes, level_start_index):
        """``value_dpt_dist`` (bs, keys, D) laid out for the operator's depth taps (``dfa3D._ext.pack_shared_dist``);
        None where that is not offered.  Valid for as long as the distribution's values do not change."""
        from .. import _ext
        bs, keys, depth = value_dpt_dist.shape
        dist = value_dpt_dist.reshape(bs, keys, 1, depth).to(self.value_proj.weight.dtype).contiguous()
        return _ext.pack_shared_dist(dist, self.get_spatial_shape_3D(spatial_shapes, depth), level_start_index)

    def sampling_locations(self, query, reference_points, spatial_shapes_3D):
        """Normalised (x, y, z) of every sampling point, (bs, Q, heads, L, points, 3): the head's learned
        offsets, divided by the level's (W, H, D), around the query's Z-anchor reference points
        (spatial_cross_attention.py:498-537).  Point p belongs to anchor p % num_Z_anchors."""
        self._check_reference_points(reference_points)
        uv, dz = projections(query, (self.sampling_offsets, self.sampling_offsets_depth))
        return self._locations(uv, dz, reference_points, spatial_shapes_3D, query.dtype)

    def _check_reference_points(self, reference_points):
        P, Z = self.num_points, reference_points.shape[2]
        if reference_points.shape[-1] != 3:
            raise ValueError("Last dim of reference_points must be 3 (x, y, depth), but get "
                             f"{reference_points.shape[-1]} instead.")
        if P % Z:
            raise ValueError(f"num_points ({P}) must be a multiple of the number of Z anchors ({Z})")

    def _locations(self, uv, dz, reference_points, spatial_shapes_3D, dtype):
        """``sampling_locations`` from the two offset layers' results (bs, Q, ...)."""
        bs, Q, _ = uv.shape
        M, L, P = self.num_heads, self.num_levels, self.num_points
        Z = reference_points.shape[2]
        uv, dz = uv.view(bs, Q, M, L, P, 2), dz.view(bs, Q, M, L, P, 1)
        if self._by_kernel(uv, dz, reference_points, spatial_shapes_3D):
            return _LocationsFunction.apply(uv, dz, reference_points, spatial_shapes_3D.contiguous())
        normalizer = spatial_shapes_3D[:, [1, 0, 2]].to(dtype)              # (W, H, D) per level
        offsets = torch.cat([uv, dz], dim=-1) / normalizer[None, None, None, :, None, :]
        anchors = reference_points[:, :, None, None, None, :, :]                   # (bs, Q, 1, 1, 1, Z, 3)
        loc = offsets.view(bs, Q, M, L, P // Z, Z, 3) + anchors
        return loc.view(bs, Q, M, L, P, 3)

    def _by_kernel(self, uv, dz, reference_points, spatial_shapes_3D, *others):
        return (ordinary(uv, dz, reference_points, *others) and all(t.is_contiguous() for t in (uv, dz, reference_points, *others))
                and not reference_points.requires_grad and reference_points.shape[:2] == uv.shape[:2] and spatial_shapes_3D.device == uv.device
                and spatial_shapes_3D.dtype == torch.int64 and spatial_shapes_3D.shape == (self.num_levels, 3))

    def _sampling(self, uv, dz, logits, reference_points, spatial_shapes_3D, dtype):
        """Locations (as ``_locations``) and attention weights from the results of the three layers of the queries.  In one kernel where a head's
        points are a power of two that a wavefront has lanes for; else the softmax is torch's."""
        bs, Q, _ = uv.shape
        M, L, P = self.num_heads, self.num_levels, self.num_points
        if L * P <= 64 and L * P & (L * P - 1) == 0 and self._by_kernel(uv, dz, reference_points, spatial_shapes_3D, logits):
            return _SamplingFunction.apply(uv.view(bs, Q, M, L, P, 2), dz.view(bs, Q, M, L, P, 1), logits.view(bs, Q, M, L, P), reference_points,
                                           spatial_shapes_3D.contiguous())
        weights = logits.view(bs, Q, M, L * P).softmax(-1).view(bs, Q, M, L, P)
        return self._locations(uv, dz, reference_points, spatial_shapes_3D, dtype), weights

    def _check_values(self, value, value_dpt_dist, spatial_shapes):
        if spatial_shapes.shape[0] != self.num_levels:
            raise ValueError(f"spatial_shapes has {spatial_shapes.shape[0]} levels, the module {self.num_levels}")
        if value_dpt_dist is None or value_dpt_dist.dim() != 3 or value_dpt_dist.shape[:2] != value.shape[:2]:
            raise ValueError("value_dpt_dist must be (bs, num_value, D)")

    def _value_side(self, value, value_dpt_dist, spatial_shapes, key_padding_mask):
        bs, num_value, _ = value.shape
        value = self.value_proj(value)
        if key_padding_mask is not None:
            value = value.masked_fill(key_padding_mask[..., None], 0.0)
        value = value.view(bs, num_value, self.num_heads, -1)
        dim_depth = value_dpt_dist.shape[2]
        dist = value_dpt_dist.reshape(bs, num_value, 1, dim_depth).to(value.dtype)
        return value, dist, self.get_spatial_shape_3D(spatial_shapes, dim_depth)

    def value_side(self, value, value_dpt_dist, spatial_shapes, key_padding_mask=None):
        """What ``forward`` makes of ``value`` (bs, keys, embed_dims), ``value_dpt_dist``, ``spatial_shapes`` and
        ``key_padding_mask`` alone."""
        self._check_values(value, value_dpt_dist, spatial_shapes)
        return self._value_side(value, value_dpt_dist, spatial_shapes, key_padding_mask)

    def _check_value_side(self, value_side, bs, value, key_padding_mask):
        """``value``: (bs, keys, embed_dims) as given to ``forward`` beside ``value_side``, or None."""
        if key_padding_mask is not None:
            raise ValueError("key_padding_mask has no effect on a value_side that is given: hand it to value_side()")
        projected, dist, shapes = value_side
        if projected.dim() != 4 or projected.shape[0] != bs or projected.shape[2] != self.num_heads:
            raise ValueError(f"value_side holds values of shape {tuple(projected.shape)}, the queries are {bs} batch elements "
                             f"for {self.num_heads} heads")
        if value is not None and value.shape[:2] != projected.shape[:2]:
            raise ValueError(f"value_side holds {tuple(projected.shape[:2])} values, value {tuple(value.shape[:2])}")
        if dist.shape[:2] != projected.shape[:2] or shapes.shape[0] != self.num_levels:
            raise ValueError("value_side is none of this module's")

    def forward(self, query, key=None, value=None, value_dpt_dist=None, identity=None, query_pos=None,
                key_padding_mask=None, reference_points=None, spatial_shapes=None, level_start_index=None,
                return_depth_score=False, packed_dist=None, value_side=None, **kwargs):
        """Arguments and results as spatial_cross_attention.py:428-583: ``query`` (bs, Q, embed_dims),
        ``value`` (bs, keys, embed_dims), ``value_dpt_dist`` (bs, keys, D), ``reference_points``
        (bs, Q, num_Z_anchors, 3) normalised, ``spatial_shapes`` (L, 2) as (h, w), ``level_start_index`` (L,).
        Returns ``(output (bs, Q, embed_dims), weight_update (bs, Q, heads, 1))``; with
        ``return_depth_score=True`` a third result, the operator's depth scores.  ``packed_dist``: what
        ``self.pack_dist(value_dpt_dist, spatial_shapes, level_start_index)`` returned for this very distribution;
        an encoder that runs several of these layers on one distribution packs once and hands it to each.
        ``value_side``: what ``self.value_side(value, value_dpt_dist, spatial_shapes, key_padding_mask)`` returned, for a
        caller that has the values before the queries; there ``value`` is batch first, and the mask is not given again."""
        given = value
        if value is None:
            value = query
        if query_pos is not None:
            query = query + query_pos
        if not self.batch_first:
            query = query.permute(1, 0, 2)
            value = value.permute(1, 0, 2)
        bs, num_query, _ = query.shape
        if value_side is None:
            self._check_values(value, value_dpt_dist, spatial_shapes)
        else:
            self._check_value_side(value_side, bs, value if given is not None else None, key_padding_mask)
        # the largest launches first: the GPU works on them while the host prepares the others
        together = getattr(self.sampling_locations, "__func__", None) is MSDeformableAttention3D_DFA3D.sampling_locations
        if together:
            self._check_reference_points(reference_points)
            uv, dz, attention_weights = projections(
                query, (self.sampling_offsets, self.sampling_offsets_depth, self.attention_weights))
        else:
            attention_weights = self.attention_weights(query)
        if value_side is None:
            value_side = self._value_side(value, value_dpt_dist, spatial_shapes, key_padding_mask)
        value, dist, spatial_shapes_3D = value_side
        if together:
            sampling_locations, attention_weights = self._sampling(uv, dz, attention_weights, reference_points, spatial_shapes_3D, query.dtype)
        else:
            attention_weights = attention_weights.view(bs, num_query, self.num_heads, self.num_levels * self.num_points).softmax(-1)
            attention_weights = attention_weights.view(bs, num_query, self.num_heads, self.num_levels, self.num_points)
            sampling_locations = self.sampling_locations(query, reference_points, spatial_shapes_3D)

        if not value.is_cuda:
            raise NotImplementedError("the DFA3D operator runs on the GPU only")
        args = (value.contiguous(), dist.contiguous(), spatial_shapes_3D, level_start_index,
                sampling_locations.contiguous(), attention_weights.contiguous(), self.im2col_step)
        depth_score = None
        if return_depth_score:
            output, depth_score = MultiScale3DDeformableAttnFunction_fp32.apply(*args)
            weight_update = (depth_score.mean(dim=-1) * attention_weights).flatten(-2).sum(dim=-1, keepdim=True)
        else:
            output, weight_update = MultiScale3DDeformableAttnWeightUpdateFunction_fp32.apply(*args, packed_dist)
        if not self.batch_first:
            output = output.permute(1, 0, 2)
        return (output, weight_update, depth_score) if return_depth_score else (output, weight_update)
