"""Performance cases of the DFA3D operator: what its users have it do, through the public entry points.

A case is a dict of plain values:
  path       "one_stage"  MultiScale3DDeformableAttnFunction: output and depth scores in one call
             "shared"     MultiScale3DDeformableAttnWeightUpdateFunction: one depth distribution for all heads
             "two_stage"  MultiScaleDepthScoreSampleFunction, then WeightedMultiScaleDeformableAttnFunction
             "plain"      MultiScaleDeformableAttnFunction: 2-D deformable attention (temporal self-attention, decoder)
             "layer"      the SpatialCrossAttention_DFA3D module around the operator, camera re-batching included
  train      False: forward under no_grad; True: forward and the gradients of everything that has one
  dtype      "f32", "bf16" (storage of value, distribution and output; locations and weights float32), "f64"
  batch      batch elements (samples x cameras); "layer": samples, each with six cameras
  queries    queries per batch element; "layer": the side of the square BEV grid
  height, width, levels   finest feature map; every further level halves it (rounding up)
  bins, points, heads, channels   depth bins, sampling points per level, heads, channels per head
  where      sampling locations: "uniform" over the map, "wide" (some outside it), "clustered" around its middle,
             "coherent" (queries in raster order over the image, a query's points a few pixels around it)
  depth      depth distributions: "soft" (softmax of normal logits) or "peaky" (one bin holds nearly everything)
  unit_sum   attention weights from a softmax (True) or drawn from [0, 1) without normalisation (False)
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.abspath("3d-deformable-attention_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from dfa3D import functional as _f  # noqa: E402
from dfa3D.modules import SpatialCrossAttention_DFA3D  # noqa: E402

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f64": torch.float64}
_CAMERAS = 6        # of a "layer"
_ANCHORS = 4        # reference points per BEV pillar of a "layer"


def _case(name, path, train, dtype, batch, queries, height, width, levels, bins, points, heads=8, channels=32,
          where="uniform", depth="soft", unit_sum=True):
    return {"name": name, "path": path, "train": train, "dtype": dtype, "batch": batch, "queries": queries,
            "height": height, "width": width, "levels": levels, "bins": bins, "points": points, "heads": heads,
            "channels": channels, "where": where, "depth": depth, "unit_sum": unit_sum}


def listed():
    return [
        # a call of the size of a unit test, forward only: latency and launches
        _case("unit_infer", "one_stage", False, "f32", 2, 100, 16, 16, 2, 16, 4),
        # checking a model's gradients in double precision, on a shape cut down for it
        _case("check_f64", "one_stage", True, "f64", 2, 400, 29, 50, 2, 32, 4, where="wide"),
        # small model: one level of 23 x 40, some points outside the image; a training step of the operator
        _case("small_train", "one_stage", True, "f32", 6, 4000, 23, 40, 1, 64, 8, where="wide"),
        # base model: four levels from 116 x 200, 15.36 M points; the headline training step
        _case("base_train", "one_stage", True, "f32", 6, 10000, 116, 200, 4, 64, 8),
        # the same with bfloat16 storage and distributions taken from measured depth
        _case("base_train_bf16", "one_stage", True, "bf16", 6, 10000, 116, 200, 4, 64, 8, depth="peaky"),
        # base model at inference, with locations as a trained model produces them
        _case("base_infer", "one_stage", False, "f32", 6, 10000, 116, 200, 4, 64, 8, where="coherent"),
        # the operands of the reference's own test, through its two separate stages
        _case("two_stage_train", "two_stage", True, "f32", 6, 9502, 116, 200, 4, 112, 8, unit_sum=False),
        # dense BEV grid with 128 bins and clustered locations, 61 M points: the largest step
        _case("dense_train", "one_stage", True, "f32", 6, 40000, 116, 200, 4, 128, 8, where="clustered"),
        # temporal self-attention over the 200 x 200 BEV map of two frames
        _case("plain_train", "plain", True, "f32", 2, 40000, 200, 200, 1, 1, 4, where="coherent"),
        # sizes that are no multiple of anything: 59 bins, 20 channels, 6 heads, odd queries and maps
        _case("ragged_train", "one_stage", True, "f32", 3, 3331, 37, 67, 3, 59, 5, heads=6, channels=20, where="wide"),
        # the whole cross-attention layer of the base model, 200 x 200 BEV queries and six cameras, training
        _case("layer_train", "layer", True, "f32", 1, 200, 116, 200, 4, 64, 8),
        # the layer of the small model at inference
        _case("layer_infer", "layer", False, "f32", 1, 150, 23, 40, 1, 64, 8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(("one_stage", "one_stage", "one_stage", "shared", "two_stage", "plain", "layer"))
    c = {"path": path, "train": rng.random() < 0.6, "dtype": "f32"}
    if path in ("one_stage", "shared", "plain"):
        c["dtype"] = rng.choice(("f32", "f32", "bf16")) if rng.random() < 0.9 else "f64"
    c["levels"] = rng.randint(1, 4)
    c["height"] = _log_int(rng, 15, 116)
    c["width"] = int(c["height"] * rng.uniform(1.3, 1.8))
    c["bins"] = 1 if path == "plain" else 16 * rng.randint(1, 8) if rng.random() < 0.6 else rng.randint(16, 128)
    c["points"] = rng.choice((4, 8)) if path == "layer" else rng.choice((2, 3, 4, 4, 5, 8, 8))
    # 32 channels in 8 heads is what the models use; other widths now and then
    usual = path == "layer" or rng.random() < 0.65
    c["heads"] = 8 if usual else rng.choice((4, 6, 8))
    c["channels"] = 32 if usual else rng.choice((16, 20, 24, 32, 40, 64))
    c["where"] = rng.choice(("uniform", "wide", "clustered", "coherent", "coherent"))
    c["depth"] = rng.choice(("soft", "soft", "peaky"))
    c["unit_sum"] = path == "layer" or rng.random() < 0.85
    if path == "layer":
        c["batch"], c["queries"] = rng.randint(1, 2), _log_int(rng, 25, 120)
        return c
    c["batch"] = rng.randint(1, 6)
    # points in total: double precision is for checks, rows that no vector width divides evenly for small models
    most = 2e5 if c["dtype"] == "f64" else 6e6 if c["channels"] in (20, 24, 40) else 2e7
    per_query = c["batch"] * c["heads"] * c["levels"] * c["points"]
    c["queries"] = _log_int(rng, 50, max(60, min(40000, most / per_query)))
    return c


def _maps(case):
    h, w, out = case["height"], case["width"], []
    for _ in range(case["levels"]):
        out.append((h, w))
        h, w = (h + 1) // 2, (w + 1) // 2
    return out


def _distribution(shape, depth, g, dev):
    if depth == "peaky":
        logits = torch.randn(shape, generator=g, device=dev)
        hot = torch.randint(0, shape[-1], shape[:-1] + (1,), generator=g, device=dev)
        logits.scatter_add_(-1, hot, torch.full(hot.shape, 8.0, device=dev))
    else:
        logits = torch.randn(shape, generator=g, device=dev).mul_(2.0)
    return logits.softmax(-1)


def _locations(case, dims, g, dev):
    B, Q, M, L, P = dims
    if case["where"] == "clustered":
        return torch.randn(B, Q, M, L, P, 3, generator=g, device=dev).mul_(0.15).add_(0.5).clamp_(-0.1, 1.1)
    if case["where"] == "coherent":
        side = max(1, int(round(Q ** 0.5)))
        q = torch.arange(Q, device=dev)
        centre = torch.stack([(q % side + 0.5) / side, (q.div(side, rounding_mode="floor") % side + 0.5) / side,
                              torch.full((Q,), 0.5, device=dev)], -1)
        loc = torch.randn(B, Q, M, L, P, 3, generator=g, device=dev)
        return loc.mul_(torch.tensor([0.02, 0.02, 0.2], device=dev)).add_(centre.view(1, Q, 1, 1, 1, 3))
    loc = torch.rand(B, Q, M, L, P, 3, generator=g, device=dev)
    return loc.mul_(1.1).sub_(0.05) if case["where"] == "wide" else loc


def _layer_state(case, g, dev):
    """A cross-attention layer with trained-like parameters, image features and depth of six cameras, and the BEV
    pillars' reference points: cameras every 60 degrees with a 70 degree view, so that a camera sees about a fifth of
    the pillars and neighbours share some."""
    M, C, D, side, bs = case["heads"], case["channels"], case["bins"], case["queries"], case["batch"]
    E, maps = M * C, _maps(case)
    S = sum(h * w for h, w in maps)
    with torch.device(dev):
        layer = SpatialCrossAttention_DFA3D(
            embed_dims=E, num_cams=_CAMERAS, bev_h=side, bev_w=side, dropout=0.0, num_head=M,
            deformable_attention=dict(type="MSDeformableAttention3D_DFA3D", embed_dims=E, num_heads=M,
                                      num_levels=case["levels"], num_points=case["points"]))
    with torch.no_grad():
        for name, p in sorted(layer.named_parameters()):
            noise = torch.randn(p.shape, generator=g, device=dev)
            if name.endswith("weight") and ("sampling_offsets" in name or "attention_weights" in name):
                p.copy_(noise * 0.03)
            elif "value_proj" in name or "output_proj" in name:
                p.copy_(noise * (E ** -0.5 if name.endswith("weight") else 0.02))
            else:
                p.add_(noise * 0.2)
    # pillars on a square of 102.4 m, cameras at its centre 1.5 m above ground, the vehicle turned and shifted a little
    turn, shift = float(torch.rand(1, generator=g, device=dev)) - 0.5, torch.rand(2, generator=g, device=dev) - 0.5
    axis = (torch.arange(side, device=dev) + 0.5) / side * 102.4 - 51.2
    py, px = torch.meshgrid(axis, axis, indexing="ij")
    px, py = (px + shift[0]).reshape(-1), (py + shift[1]).reshape(-1)
    z = torch.linspace(-1.0, 3.0, _ANCHORS, device=dev)
    yaw = turn + torch.arange(_CAMERAS, device=dev) * (2 * math.pi / _CAMERAS)
    ahead = px * torch.cos(yaw)[:, None] + py * torch.sin(yaw)[:, None]                 # (cameras, pillars)
    aside = py * torch.cos(yaw)[:, None] - px * torch.sin(yaw)[:, None]
    near, half = ahead.clamp(min=0.1), math.tan(math.radians(35.0))
    u = (0.5 + aside / near / (2 * half))[..., None].expand(-1, -1, _ANCHORS)
    v = 0.5 + (1.5 - z) / near[..., None] / (2 * half * maps[0][0] / maps[0][1])
    deep = (near / 75.0)[..., None].expand(-1, -1, _ANCHORS)
    ref = torch.stack([u, v, deep], -1)[:, None].expand(-1, bs, -1, -1, -1).contiguous()
    mask = (ahead[..., None] > 1.0) & (u > 0) & (u < 1) & (v > 0) & (v < 1)
    grad = case["train"]
    features = torch.randn(_CAMERAS, S, bs, E, generator=g, device=dev).requires_grad_(grad)
    state = {
        "layer": layer if grad else layer.eval(),
        "query": torch.randn(bs, side * side, E, generator=g, device=dev).requires_grad_(grad),
        "query_pos": torch.randn(bs, side * side, E, generator=g, device=dev).mul_(0.1),
        "features": features,
        "dist": _distribution((_CAMERAS, S, bs, D), case["depth"], g, dev).requires_grad_(grad),
        "ref": ref, "mask": mask[:, None].expand(-1, bs, -1, -1).contiguous(),
        "shapes": torch.tensor(maps, device=dev),
        "grad_out": torch.randn(bs, side * side, E, generator=g, device=dev),
    }
    if grad:
        state["leaves"] = [state["query"], features, state["dist"]] + [p for _, p in sorted(layer.named_parameters())]
    return state


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed))
    maps = _maps(case)
    starts, acc = [], 0
    for h, w in maps:
        starts.append(acc)
        acc += h * w
    S, M, C, D = acc, case["heads"], case["channels"], case["bins"]
    start = torch.tensor(starts, dtype=torch.int64, device=dev)
    if case["path"] == "layer":
        return dict(_layer_state(case, g, dev), path="layer", train=case["train"], start=start)
    B, Q, L, P = case["batch"], case["queries"], case["levels"], case["points"]
    store = _DTYPES[case["dtype"]]
    aux = torch.float64 if case["dtype"] == "f64" else torch.float32
    plain = case["path"] == "plain"
    value = torch.randn(B, S, M, C, generator=g, device=dev).to(store)
    dist = None
    if not plain:
        dist = _distribution((B, S, 1 if case["path"] == "shared" else M, D), case["depth"], g, dev).to(store)
    loc = _locations(case, (B, Q, M, L, P), g, dev).to(aux)
    loc = loc[..., :2].contiguous() if plain else loc
    if case["unit_sum"]:
        attn = torch.randn(B, Q, M, L * P, generator=g, device=dev).softmax(-1).view(B, Q, M, L, P).to(aux)
    else:
        attn = torch.rand(B, Q, M, L, P, generator=g, device=dev).to(aux)
    state = {"path": case["path"], "train": case["train"], "start": start, "value": value, "dist": dist, "loc": loc,
             "attn": attn, "shapes": torch.tensor([[h, w] if plain else [h, w, D] for h, w in maps],
                                                  dtype=torch.int64, device=dev)}
    if case["train"]:
        state["leaves"] = [t.requires_grad_() for t in (value, dist, loc, attn) if t is not None]
        state["grad_out"] = torch.randn(B, Q, M * C, generator=g, device=dev).to(store)
        if case["path"] == "shared":
            state["grad_update"] = torch.randn(B, Q, M, 1, generator=g, device=dev).to(aux)
    return state


def _forward(s):
    if s["path"] == "layer":
        return (s["layer"](s["query"], s["features"], s["features"], query_pos=s["query_pos"],
                           spatial_shapes=s["shapes"], reference_points_cam=s["ref"], bev_mask=s["mask"],
                           level_start_index=s["start"], value_dpt_dist=s["dist"]),)
    if s["path"] == "one_stage":
        return _f.MultiScale3DDeformableAttnFunction.apply(
            s["value"], s["dist"], s["shapes"], s["start"], s["loc"], s["attn"], 64)
    if s["path"] == "shared":
        return _f.MultiScale3DDeformableAttnWeightUpdateFunction.apply(
            s["value"], s["dist"], s["shapes"], s["start"], s["loc"], s["attn"], 64)
    if s["path"] == "plain":
        return (_f.MultiScaleDeformableAttnFunction.apply(
            s["value"], s["shapes"], s["start"], s["loc"], s["attn"], 64),)
    score = _f.MultiScaleDepthScoreSampleFunction.apply(s["dist"], s["shapes"], s["start"], s["loc"], 64)
    out = _f.WeightedMultiScaleDeformableAttnFunction.apply(
        s["value"], s["shapes"][:, :2].contiguous(), s["start"], s["loc"][..., :2].contiguous(), s["attn"], score, 64)
    return out, score


def run(state):
    if not state["train"]:
        with torch.no_grad():
            return _forward(state)
    out = _forward(state)
    if state["path"] == "shared":
        grads = torch.autograd.grad(out, state["leaves"], (state["grad_out"], state["grad_update"]))
    else:
        grads = torch.autograd.grad(out[0], state["leaves"], state["grad_out"])
    return tuple(t.detach() for t in out) + tuple(grads)


def work(case):
    """Every input read once, every output written once; arithmetic on the sampled rows and, in a layer, the dense
    projections."""
    e = {"f32": 4, "bf16": 2, "f64": 8}[case["dtype"]]
    a = 8 if case["dtype"] == "f64" else 4
    S = sum(h * w for h, w in _maps(case))
    M, C, D = case["heads"], case["channels"], case["bins"]
    LP, train = case["levels"] * case["points"], case["train"]
    if case["path"] == "layer":
        E, Q, bs = M * C, case["queries"] ** 2, case["batch"]
        features, dist, rows = bs * _CAMERAS * S * E, bs * _CAMERAS * S * D, bs * Q * E
        seen = bs * Q * 1.2                                     # pillars x cameras that see them
        params = E * (E + E + 4 * M * LP) + 4 * M * LP + 2 * E
        nbytes = 4 * (features + dist + 3 * rows + bs * _CAMERAS * Q * _ANCHORS * 3 + params) + bs * _CAMERAS * Q * _ANCHORS
        flops = 2 * E * E * (bs * _CAMERAS * S + bs * Q) + 2 * E * 4 * M * LP * seen + 8 * seen * M * LP * C
        if train:
            nbytes += 4 * (features + dist + 2 * rows + params)
            flops *= 3
        return {"bytes": nbytes, "flops": flops}
    B, Q = case["batch"], case["queries"]
    n = B * Q * M * LP
    plain, shared = case["path"] == "plain", case["path"] == "shared"
    whole = B * S * (M * C + (0 if plain else D if shared else M * D))
    # few points on a large map read four rows and eight bins each, not all of it; gradients are written whole
    sampled = min(B * S * M * C, 4 * n * C) + (0 if plain else min(B * S * D * (1 if shared else M), 8 * n))
    coords = 2 if plain else 3
    score = 0 if plain or shared else 4 * n
    nbytes = e * (sampled + B * Q * M * C + score) + a * ((coords + 1) * n + (B * Q * M if shared else 0))
    flops = n * (8 * C + (0 if plain else 12))
    if train:
        nbytes += e * (whole + B * Q * M * C) + a * ((coords + 1) * n + (B * Q * M if shared else 0))
        flops *= 3
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["dtype"] == "f64":
        return {"rel": 1e-11}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2}
    # in a layer the float32 rounding of the projections goes through the sampling before the sums are formed
    return {"rel": 1e-4 if case["path"] == "layer" else 1e-5}
