"""What a cross-attention layer gathers in one launch against the gathers one by one, the counts that come with the hits against the tensor operations, and
the level table: odd and wide rows, unaligned bases, query counts around a workgroup's, cameras that see nothing; all of it moves or counts, and one sum of
two numbers, so results are equal to the bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _offset(shape, dtype, by):
    n = torch.Size(shape).numel()
    return torch.randn(n + by, dtype=dtype, device="cuda")[by:].view(shape)


@pytest.mark.parametrize("cams,bs,Nq,E,R,dtype,by", [
    (6, 1, 333, 256, 12, torch.float32, 0), (3, 2, 70, 64, 9, torch.float32, 0), (2, 3, 41, 30, 12, torch.float32, 0), (2, 1, 41, 6, 3, torch.float64, 0),
    (2, 2, 50, 32, 12, torch.float32, 1), (1, 1, 1, 4, 4, torch.float64, 0), (70, 20, 9, 8, 3, torch.float32, 0)])
@pytest.mark.parametrize("added", [True, False], ids=["plus", "alone"])
def test_queries_and_points_in_one_launch(cams, bs, Nq, E, R, dtype, by, added):
    from dfa3D.rebatch import RebatchQueriesFunction, camera_index, rebatch_combine, rebatch_gather, rebatch_queries
    torch.manual_seed(Nq)
    hit = torch.rand(cams, Nq, device="cuda") < 0.3
    if cams > 1:
        hit[1] = False
    index, pos, _ = camera_index(hit)
    src, plus, ref = _offset((bs, Nq, E), dtype, by), _offset((bs, Nq, E), dtype, 0) if added else None, _offset((cams, bs, Nq, R), dtype, by)
    src.view(-1)[0], ref.view(-1)[-1] = float("nan"), float("-inf")
    total = src + plus if added else src
    want, want_ref = rebatch_gather(total, index), rebatch_gather(ref, index, per_camera=True, pad=-64.0)
    got, got_ref = rebatch_queries(src, plus, ref, index, -64.0)
    bits = torch.int32 if dtype == torch.float32 else torch.int64
    assert torch.equal(got.view(bits), want.view(bits)) and torch.equal(got_ref.view(bits), want_ref.view(bits))
    leaves = [t.requires_grad_() for t in (src.detach(), plus) if t is not None]
    out, points = RebatchQueriesFunction.apply(leaves[0], leaves[1] if added else None, ref, index, pos, -64.0)
    assert out.requires_grad and not points.requires_grad
    g = torch.randn_like(out)
    for grad in torch.autograd.grad(out, leaves, g):
        assert torch.equal(grad, rebatch_combine(g, pos))
    # the combine, cameras in order, against the tensor operations
    want = torch.zeros(bs, Nq, E, dtype=dtype, device="cuda")
    for i in range(cams):
        on = pos[i] >= 0
        want[:, on] += g[:, i, pos[i][on].long()]
    assert torch.equal(rebatch_combine(g, pos), want)


@pytest.mark.parametrize("cams,bs,Nq,Z,share", [(6, 1, 22500, 4, 0.1), (3, 2, 1023, 4, 0.5), (2, 3, 1024, 3, 0.3), (1, 1, 1025, 8, 1.0), (5, 1, 70, 2, 0.0),
                                                (1, 1, 1, 1, 1.0), (2, 4, 2 ** 16, 1, 0.3), (2, 4, 2 ** 16 + 1, 1, 0.3), (1024, 1, 3, 4, 0.2), (1025, 1, 3, 4, 0.2)])
def test_counts_with_the_hits(cams, bs, Nq, Z, share):
    from dfa3D.rebatch import camera_hits, camera_hits_counted, camera_index
    mask = torch.rand(cams, bs, Nq, Z, generator=torch.Generator().manual_seed(Nq)) < share
    hit, scale, counted = camera_hits_counted(mask.cuda())
    want_hit, want_scale = camera_hits(mask)              # tensor operations
    assert torch.equal(hit.cpu(), want_hit) and torch.equal(scale.cpu(), want_scale)
    got, want = camera_index(hit, counted), camera_index(want_hit)
    assert got[2] == want[2] and torch.equal(got[0].cpu(), want[0]) and torch.equal(got[1].cpu(), want[1])
    assert torch.equal(counted[0].view(cams, -1).sum(1).cpu(), want_hit.sum(1))


def test_counts_of_other_masks():
    from dfa3D.rebatch import camera_hits_counted
    mask = torch.rand(3, 2, 50, 4) < 0.3
    for m in (mask, mask.cuda().long()):                  # tensor operations
        hit, scale, counted = camera_hits_counted(m)
        assert torch.equal(hit.cpu(), (mask.sum(-1) > 0)[:, 0]) and (counted is None) == (not m.is_cuda or not hit.is_contiguous())


@pytest.mark.parametrize("L", [1, 4, 30])
def test_level_table(L):
    from dfa3D.modules import MSDeformableAttention3D_DFA3D
    shapes = torch.randint(1, 500, (L, 2))
    want = torch.cat([shapes, torch.full((L, 1), 59)], -1)
    table = MSDeformableAttention3D_DFA3D.get_spatial_shape_3D
    for s in (shapes, shapes.cuda(), shapes.cuda().t().contiguous().t()):
        assert torch.equal(table(s, 59).cpu(), want)


def test_layer_with_positions_in_other_forms():
    """Positions that the gather may not add (broadcast, transposed, a subclass) and those it adds give the same layer, gradients included."""
    from dfa3D.modules import SpatialCrossAttention_DFA3D
    torch.manual_seed(0)
    cams, bs, Nq, E, maps = 2, 2, 64, 32, [(6, 9)]
    layer = SpatialCrossAttention_DFA3D(embed_dims=E, num_cams=cams, bev_h=8, bev_w=8, dropout=0.0, num_head=4,
                                        deformable_attention=dict(embed_dims=E, num_heads=4, num_levels=1, num_points=4)).cuda()
    query, pos = (torch.randn(bs, Nq, E, device="cuda", requires_grad=True) for _ in range(2))
    feats, dist = torch.randn(cams, 54, bs, E, device="cuda"), torch.rand(cams, 54, bs, 8, device="cuda").softmax(-1)
    args = dict(spatial_shapes=torch.tensor(maps, device="cuda"), level_start_index=torch.tensor([0], device="cuda"),
                reference_points_cam=torch.rand(cams, bs, Nq, 4, 3, device="cuda"), bev_mask=torch.rand(cams, bs, Nq, 4, device="cuda") < 0.2,
                value_dpt_dist=dist)

    def run(q, p):
        out = layer(q, feats, feats, query_pos=p, **args)
        return (out, *torch.autograd.grad(out, (query, pos), torch.ones_like(out)))

    want = run(query, pos)
    for q, p in ((query.transpose(0, 1).contiguous().transpose(0, 1), pos), (query, pos.transpose(1, 2).contiguous().transpose(1, 2)),
                 (query, pos.as_subclass(type("Sub", (torch.Tensor,), {})))):
        for g, w in zip(run(q, p), want):
            torch.testing.assert_close(g.float(), w, rtol=1e-5, atol=1e-5)
    few = pos[:1].detach().expand(bs, Nq, E)
    torch.testing.assert_close(layer(query, feats, feats, query_pos=few, **args), layer(query, feats, feats, query_pos=pos[:1].detach(), **args), rtol=0, atol=0)


@pytest.mark.parametrize("Nq", [1023, 1024, 1025, 1026, 1027, 3073, 4099])
@pytest.mark.parametrize("by", [0, 1, 2, 3])
def test_lists_of_hits_at_any_byte(Nq, by):
    """A block counts the hits before its own by whole words, and the bytes around them."""
    from dfa3D.rebatch import camera_index
    g = torch.Generator().manual_seed(Nq)
    hit = torch.rand(3, Nq, generator=g) < 0.4
    on = torch.zeros(3 * Nq + by, dtype=torch.bool, device="cuda")[by:].view(3, Nq).copy_(hit)
    got, want = camera_index(on), camera_index(hit)
    assert got[2] == want[2] and torch.equal(got[0].cpu(), want[0]) and torch.equal(got[1].cpu(), want[1])
