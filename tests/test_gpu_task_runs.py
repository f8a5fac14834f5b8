"""The forward's tasks, which each row slot of a unit has side by side: slots that get unequal numbers of them, units in three rounds, a
run that LDS has no room to pad; and the two taps of a distribution as weights of a pair of bins, where what is no tap must not be felt."""
import pytest
import torch

from forms import tiny_case
from test_gpu_parity import F32_FWD, _as_inputs, _dev

pytestmark = pytest.mark.gpu

LEVELS = ((9, 13), (5, 7), (3, 4), (2, 2))


# enough queries that a wavefront keeps as many units as it has lanes for
@pytest.mark.parametrize("L,P,C,Q", [(3, 7, 32, 1031), (3, 7, 16, 1031), (1, 9, 32, 2051), (1, 17, 64, 1025), (1, 19, 128, 1027), (1, 13, 20, 1367),
                                     (4, 11, 32, 519), (1, 65, 32, 130)])
@pytest.mark.parametrize("levels", [LEVELS, ((40, 61), (20, 31), (10, 16), (5, 8))], ids=["in LDS", "from memory"])
def test_unequal_runs(oracle, L, P, C, Q, levels):
    from dfa3D import _ext
    dev = _dev()
    t = _as_inputs(tiny_case(seed=17 * P + C, B=2, M=2, C=C, D=6, Q=Q, P=P, levels=levels[:L]))
    args = [t[k].float() if t[k].is_floating_point() else t[k] for k in
            ("value", "value_dpt_dist", "spatial_shapes", "level_start_index", "sampling_locations", "attention_weights")]
    want, want_score = oracle.dfa3d_forward(*args)
    got, score = _ext.dfa3d_fused_forward(*(x.to(dev) for x in args), 64, need_depth_score=True)
    torch.testing.assert_close(got.cpu(), want, **F32_FWD)
    torch.testing.assert_close(score.cpu(), want_score, **F32_FWD)


@pytest.mark.parametrize("D,extent", [(2, 2), (3, 2), (7, 7), (7, 4), (1, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64], ids=["fp32", "bf16", "fp64"])
def test_bins_that_are_no_taps(oracle, D, extent, dtype):
    """Depths on both sides of the first and of the last bin; bins beyond a level's depth extent hold NaN and infinities."""
    from dfa3D import _ext
    dev = _dev()
    t = _as_inputs(tiny_case(seed=D, B=1, M=2, C=8, D=D, Q=64, P=4, levels=((5, 6), (3, 3))))
    aux = torch.float64 if dtype == torch.float64 else torch.float32
    dist = t["value_dpt_dist"].to(dtype)
    clean = dist.clone()
    clean[..., extent:] = 0
    dist[..., extent:] = torch.tensor([float("nan"), float("inf"), float("-inf"), float("nan"), float("inf")], dtype=dtype)[:D - extent]
    sh = t["spatial_shapes"].clone()
    sh[:, 2] = extent
    loc = t["sampling_locations"].to(aux)
    edges = torch.linspace(-0.75, extent + 0.25, 64, dtype=aux) / extent
    loc[..., 2] = edges.view(1, -1, 1, 1, 1)
    rest = [loc, t["attention_weights"].to(aux)]
    value = t["value"].to(dtype)
    want, want_score = oracle.dfa3d_forward(value.to(aux), clean.to(aux), sh, t["level_start_index"], *rest)
    got, score = _ext.dfa3d_fused_forward(*(x.to(dev) for x in (value, dist, sh, t["level_start_index"], *rest)), 64, need_depth_score=True)
    tol = {torch.float32: F32_FWD, torch.float64: dict(rtol=1e-10, atol=1e-11), torch.bfloat16: dict(rtol=2 ** -8, atol=1e-5)}[dtype]
    torch.testing.assert_close(got.cpu().to(aux), want, **tol)
    torch.testing.assert_close(score.cpu().to(aux), want_score, **tol)


@pytest.mark.parametrize("M,levels", [(2, ((5, 6), (3, 3))), (3, ((4, 6), (2, 3))), (1, ((5, 7), (3, 3))), (1, ((5, 7), (2, 3)))])
@pytest.mark.parametrize("D", [2, 3, 7, 8, 59])
@pytest.mark.parametrize("first", [0, 1])
def test_pairs_of_2_byte_bins(oracle, M, levels, D, first):
    """Batch elements whose distributions begin and end on words and ones that do not, in memory of NaN; half of the points at the ends of the last
    pixel's distribution."""
    from dfa3D import _ext
    dev = _dev()
    t = _as_inputs(tiny_case(seed=D + M, B=3, M=M, C=8, D=D, Q=64, P=4, levels=levels))
    value, dist, attn, loc = t["value"].bfloat16(), t["value_dpt_dist"].bfloat16(), t["attention_weights"].float(), t["sampling_locations"].float()
    for l, (h, w) in enumerate(levels):
        loc[:, ::2, :, l, :, 0], loc[:, ::2, :, l, :, 1] = (w - 0.4) / w, (h - 0.6) / h
    loc[:, ::4, ..., 2] = torch.linspace(-0.3, 0.7, 16).view(1, -1, 1, 1, 1) / D
    loc[:, 2::4, ..., 2] = 1 + torch.linspace(-0.9, 0.3, 16).view(1, -1, 1, 1, 1) / D
    memory = torch.full((dist.numel() + 16,), float("nan"), dtype=torch.bfloat16, device=dev)
    given = memory[8 + first:8 + first + dist.numel()].view(dist.shape).copy_(dist)
    want, want_score = oracle.dfa3d_forward(value.float(), dist.float(), t["spatial_shapes"], t["level_start_index"], loc, attn)
    got, score = _ext.dfa3d_fused_forward(value.to(dev), given, t["spatial_shapes"].to(dev), t["level_start_index"].to(dev), loc.to(dev), attn.to(dev), 64,
                                          need_depth_score=True)
    # one rounding to bfloat16 is 2^-9 of a number; another 2^-9 for float32 sums in another order, which may tip it the other way
    torch.testing.assert_close(got.cpu().float(), want, rtol=2 ** -8, atol=1e-5)
    torch.testing.assert_close(score.cpu().float(), want_score, rtol=2 ** -8, atol=1e-5)


def _forward_against_oracle(oracle, C, levels, call, dtype, Q, P, B=1):
    from dfa3D import _ext
    dev = _dev()
    t = _as_inputs(tiny_case(seed=C + len(levels), B=B, M=2, C=C, D=4, Q=Q, P=P, levels=levels))
    value, dist = (t[k].to(dtype) for k in ("value", "value_dpt_dist"))
    sh, lsi, loc, attn = t["spatial_shapes"], t["level_start_index"], t["sampling_locations"].float(), t["attention_weights"].float()
    if call == "packed":
        dist = dist[:, :, :1].contiguous()
    want, score = oracle.dfa3d_forward(value.float(), dist.float().expand(-1, -1, 2, -1).contiguous(), sh, lsi, loc, attn)
    on = [x.to(dev) for x in (value, dist, sh, lsi, loc, attn)]
    if call in ("one stage", "packed"):
        packed = _ext.pack_shared_dist(*on[1:4]) if call == "packed" else None
        got = _ext.dfa3d_fused_forward(*on, 64, need_depth_score=False, packed_dist=packed)[0]
    else:
        from dfa3D import functional
        xy, sh2 = on[4][..., :2].contiguous(), on[2][:, :2].contiguous()
        if call == "plain":
            got = functional.MultiScaleDeformableAttnFunction.apply(on[0], sh2, on[3], xy, on[5], 64)
            want = oracle.dfa3d_forward(value.float(), torch.ones_like(t["value_dpt_dist"][..., :1]).float(),
                                        torch.cat([sh[:, :2], torch.ones_like(sh[:, :1])], 1), lsi,
                                        torch.cat([loc[..., :2], torch.full_like(loc[..., :1], 0.5)], -1), attn)[0]
        else:
            given = score.to(dtype)
            got = functional.WeightedMultiScaleDeformableAttnFunction.apply(on[0], sh2, on[3], xy, on[5], given.to(dev), 64)
    # bfloat16: the output's own rounding, and that of the scores that are handed over
    tol = F32_FWD if dtype == torch.float32 else dict(rtol=2 ** -7, atol=2 ** -7)
    torch.testing.assert_close(got.float().cpu(), want, **tol)


# value rows of one (batch, head) on both sides of 2 MB, where the order of a unit's tasks changes: 128 and 64 channels, 4096 and 8192 keys
@pytest.mark.parametrize("C,levels", [(128, ((64, 63), (8, 8))), (128, ((64, 63), (8, 8), (1, 1))), (64, ((91, 90),)), (64, ((91, 90), (2, 2)))])
@pytest.mark.parametrize("call", ["one stage", "packed", "scores", "plain"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_order_of_tasks(oracle, C, levels, call, dtype):
    _forward_against_oracle(oracle, C, levels, call, dtype, 1301, 7)


# the same with several slots a unit on both sides: one unit of 128 channels a wavefront, two of 64, and bfloat16 rows of half the bytes
@pytest.mark.parametrize("dtype,C,Q,levels", [(torch.float32, 128, 400, ((64, 64),)), (torch.float32, 128, 400, ((64, 64), (1, 1))),
                                              (torch.bfloat16, 128, 400, ((91, 90), (1, 2))), (torch.bfloat16, 128, 400, ((91, 90), (3, 1))),
                                              (torch.bfloat16, 64, 1301, ((128, 128),)), (torch.bfloat16, 64, 1301, ((128, 128), (1, 1)))])
@pytest.mark.parametrize("call", ["one stage", "packed", "scores", "plain"])
def test_order_of_tasks_where_units_have_several_slots(oracle, dtype, C, Q, levels, call):
    _forward_against_oracle(oracle, C, levels, call, dtype, Q, 7)


# runs from memory: above 2 MB, so that 2, 4, 8 and 16 slots share a unit, with the shapes of test_unequal_runs
@pytest.mark.parametrize("L,P,C,Q", [(3, 7, 32, 1031), (3, 7, 16, 1031), (1, 9, 32, 2051), (1, 17, 64, 1025), (1, 19, 128, 1027), (1, 13, 20, 1367),
                                     (4, 11, 32, 519), (1, 65, 32, 130)])
@pytest.mark.parametrize("call", ["one stage", "packed", "scores", "plain"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_unequal_runs_of_large_maps(oracle, L, P, C, Q, call, dtype):
    rows = (2 << 20) // (C * (4 if dtype == torch.float32 else 2)) + 1
    _forward_against_oracle(oracle, C, (((rows + 126) // 127, 127),) + LEVELS[1:L], call, dtype, Q, P, B=2)


# value rows of one (batch, head) on both sides of 1.5 MB, above which units of four points have their first operands asked for before the level table:
# 12288 rows of 32 channels, 6144 of 64, 1512 of 260 (two passes over the channels)
@pytest.mark.parametrize("C,levels,P", [(32, ((96, 128),), 4), (32, ((97, 128),), 4), (32, ((96, 128), (1, 1)), 2), (64, ((64, 97), (2, 1), (1, 1), (1, 1)), 1),
                                        (260, ((36, 42),), 4), (260, ((37, 42),), 4), (28, ((120, 128),), 4), (32, ((97, 128),), 3)])
@pytest.mark.parametrize("Q", [1, 301, 8201])
@pytest.mark.parametrize("scores", [False, True])
def test_units_of_four_points(oracle, C, levels, P, Q, scores):
    """Plain attention and given scores, from one unit per wavefront up to sixteen."""
    from dfa3D import functional
    dev = _dev()
    t = _as_inputs(tiny_case(seed=C + P + Q, B=1, M=2, C=C, D=2, Q=Q, P=P, levels=levels))
    value, dist, sh, lsi, loc, attn = (t[k].float() if t[k].is_floating_point() else t[k] for k in
                                       ("value", "value_dpt_dist", "spatial_shapes", "level_start_index", "sampling_locations", "attention_weights"))
    if not scores:
        dist, sh, loc = torch.ones_like(dist[..., :1]), torch.cat([sh[:, :2], torch.ones_like(sh[:, :1])], 1), torch.cat([loc[..., :2], torch.full_like(loc[..., :1], 0.5)], -1)
    want, score = oracle.dfa3d_forward(value, dist.contiguous(), sh, lsi, loc, attn)
    v, s2, start, xy, a = (x.to(dev) for x in (value, sh[:, :2].contiguous(), lsi, loc[..., :2].contiguous(), attn))
    got = (functional.WeightedMultiScaleDeformableAttnFunction.apply(v, s2, start, xy, a, score.to(dev), 64) if scores else
           functional.MultiScaleDeformableAttnFunction.apply(v, s2, start, xy, a, 64))
    torch.testing.assert_close(got.cpu(), want, **F32_FWD)


@pytest.mark.parametrize("L", [1, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("packed", [False, True])
def test_levels_four_at_a_time(oracle, L, packed):
    """Tables of one to sixteen levels; a level that does not fit the keys or bins adds nothing, as with weights of zero."""
    from dfa3D import _ext
    dev = _dev()
    t = _as_inputs(tiny_case(seed=L, B=2, M=2, C=16, D=5, Q=37, P=3, levels=tuple((3 + l % 4, 2 + l % 3) for l in range(L))))
    value, dist, sh, lsi, loc, attn = (t[k].float() if t[k].is_floating_point() else t[k] for k in
                                       ("value", "value_dpt_dist", "spatial_shapes", "level_start_index", "sampling_locations", "attention_weights"))
    if packed:
        dist = dist[:, :, :1].contiguous()
    bad, bad_lsi, kept = sh.clone(), lsi.clone(), attn.clone()
    for l, column, number in ((1, 0, 2 ** 32 + 3), (4, 2, 6), (7, 1, -2), (8, 0, 2 ** 31), (15, 2, 2 ** 32 + 5)):
        if l < L:
            bad[l, column] = number
            kept[:, :, :, l] = 0
    if L > 2:
        bad_lsi[2] = -1
        kept[:, :, :, 2] = 0
    want, _ = oracle.dfa3d_forward(value, dist.expand(-1, -1, 2, -1).contiguous(), sh, lsi, loc, kept)
    on = [x.to(dev) for x in (value, dist, bad, bad_lsi, loc, attn)]
    got = _ext.dfa3d_fused_forward(*on, 64, need_depth_score=False, packed_dist=_ext.pack_shared_dist(*on[1:4]) if packed else None)[0]
    torch.testing.assert_close(got.cpu(), want, **F32_FWD)


@pytest.mark.parametrize("L", [1, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("map_rows", [95, 97])
@pytest.mark.parametrize("Q", [37, 1301])
def test_packed_levels_of_large_maps(oracle, L, map_rows, Q):
    """A packed float32 distribution on both sides of 1.5 MB of value rows, above which each wavefront reads the levels' sizes itself: as above, and
    with levels that share keys, whose cells are more than the packed table holds."""
    from dfa3D import _ext
    dev = _dev()
    levels = ((map_rows, 127),) + tuple((3 + l % 4, 2 + l % 3) for l in range(1, L))
    t = _as_inputs(tiny_case(seed=L, B=2, M=2, C=32, D=5, Q=Q, P=3, levels=levels))
    value, dist, sh, lsi, loc, attn = (t[k].float() if t[k].is_floating_point() else t[k] for k in
                                       ("value", "value_dpt_dist", "spatial_shapes", "level_start_index", "sampling_locations", "attention_weights"))
    dist = dist[:, :, :1].contiguous()
    both = dist.expand(-1, -1, 2, -1).contiguous()
    bad, kept = sh.clone(), attn.clone()
    for l, column, number in ((2, 0, 2 ** 32 + 3), (4, 2, 6), (7, 1, -2), (8, 0, 2 ** 31), (15, 2, 2 ** 32 + 5)):
        if l < L:
            bad[l, column] = number
            kept[:, :, :, l] = 0
    shared, from_zero = sh[:1].expand(L, -1).contiguous(), torch.zeros_like(lsi)
    for given, shapes, start, weights in ((bad, sh, lsi, kept), (shared, shared, from_zero, attn)):
        want, _ = oracle.dfa3d_forward(value, both, shapes, start, loc, weights)
        on = [x.to(dev) for x in (value, dist, given, start, loc, attn)]
        got = _ext.dfa3d_fused_forward(*on, 64, need_depth_score=False, packed_dist=_ext.pack_shared_dist(*on[1:4]))[0]
        torch.testing.assert_close(got.cpu(), want, **F32_FWD)


@pytest.mark.parametrize("D", [2, 31, 64, 255, 256, 257, 600])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_packed_table_as_laid_out(D, dtype):
    """Every cell and bin against the four pixels around it: rows of cells of one run and of several, an empty level, a map of one pixel."""
    from dfa3D import _ext
    dev = _dev()
    levels, B = ((5, 130), (1, 1), (7, 3)), 3
    S = sum(h * w for h, w in levels) + 4
    dist = torch.rand(B, S, 1, D, generator=torch.Generator().manual_seed(D)).to(dtype)
    sh = torch.tensor([(h, w, D) for h, w in levels] + [(S + 1, 2, D)])                  # the last does not fit: empty
    start = [0, 650, 651, 0]
    got = _ext.pack_shared_dist(dist.to(dev), sh.to(dev), torch.tensor(start).to(dev))
    want = []
    for (h, w), s in zip(levels + ((0, 0),), start):
        m = torch.nn.functional.pad(dist[:, s:s + h * w, 0].reshape(B, h, w, D), (0, 0, 1, 1, 1, 1))
        four = torch.stack([m[:, :-1, :-1], m[:, :-1, 1:], m[:, 1:, 1:], m[:, 1:, :-1]], -1)
        want.append(four.reshape(B, (h + 1) * (w + 1) * D * 4))
    want = torch.cat(want, 1)
    assert torch.equal(got.view(dtype)[:want.numel()].cpu(), want.view(-1))
