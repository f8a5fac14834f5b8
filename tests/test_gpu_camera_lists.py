"""The re-batching lists made on the GPU against the plain tensor operations: query counts around the blocks that rank them,
cameras that see nothing or everything, masks of any anchor count and alignment."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cams,bs,Nq,Z,share", [(6, 1, 22500, 4, 0.2), (1, 1, 1, 1, 1.0), (3, 2, 1023, 4, 0.5), (2, 3, 1024, 3, 0.3),
                                                (6, 2, 1025, 8, 0.1), (4, 1, 40000, 4, 1.0), (5, 1, 70, 2, 0.0), (7, 2, 3001, 5, 0.02)])
def test_hits_scale_and_lists(cams, bs, Nq, Z, share):
    from dfa3D.rebatch import camera_hits, camera_index
    g = torch.Generator().manual_seed(Nq + Z)
    mask = torch.rand(cams, bs, Nq, Z, generator=g) < share
    if cams > 2:
        mask[1] = False                                   # a camera that sees nothing
    hit, scale = camera_hits(mask.cuda())
    want_hit, want_scale = camera_hits(mask)              # tensor operations
    assert torch.equal(hit.cpu(), want_hit) and torch.equal(scale.cpu(), want_scale)
    # a mask that starts between words
    odd = torch.zeros(mask.numel() + 1, dtype=torch.bool, device="cuda")[1:].view(mask.shape).copy_(mask)
    hit2, scale2 = camera_hits(odd)
    assert torch.equal(hit2, hit) and torch.equal(scale2, scale)
    index, pos, max_len = camera_index(hit)
    want_index, want_pos, want_len = camera_index(want_hit)
    assert max_len == want_len and torch.equal(index.cpu(), want_index) and torch.equal(pos.cpu(), want_pos)
    counted = camera_hits(mask.cuda().long())             # numbers instead of truth values: as before
    assert torch.equal(counted[0], hit) and torch.equal(counted[1], scale)


@pytest.mark.parametrize("E", [12, 7])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["fp32", "fp64"])
def test_gather_pads_with_what_it_is_told(E, dtype):
    from dfa3D.rebatch import rebatch_gather
    index = torch.tensor([[0, 3, 4, -1], [2, -1, -1, -1]], dtype=torch.int32, device="cuda")
    src = torch.randn(2, 3, 5, E, dtype=dtype, device="cuda")
    zeros, far = rebatch_gather(src, index, per_camera=True), rebatch_gather(src, index, per_camera=True, pad=-64.0)
    on = (index >= 0)[None, :, :, None].expand_as(zeros)
    assert torch.equal(zeros[on], far[on]) and (zeros[~on] == 0).all() and (far[~on] == -64).all()


def test_layer_does_not_depend_on_the_padding(monkeypatch):
    """Results and gradients with the padded queries' samples outside the map and on its first pixels."""
    from dfa3D.modules import SpatialCrossAttention_DFA3D, spatial_cross_attention
    torch.manual_seed(0)
    dev, cams, bs, Nq, E, maps = "cuda", 3, 2, 300, 64, [(9, 14), (5, 7)]
    keys = sum(h * w for h, w in maps)
    layer = SpatialCrossAttention_DFA3D(embed_dims=E, num_cams=cams, bev_h=15, bev_w=20, dropout=0.0, num_head=4, use_empty=True,
                                        deformable_attention=dict(embed_dims=E, num_heads=4, num_levels=2, num_points=4)).to(dev)
    for p in layer.parameters():
        torch.nn.init.normal_(p, std=0.1)
    query = torch.randn(bs, Nq, E, device=dev, requires_grad=True)
    feats = torch.randn(cams, keys, bs, E, device=dev, requires_grad=True)
    dist = torch.rand(cams, keys, bs, 8, device=dev).softmax(-1).requires_grad_()
    mask = torch.rand(cams, bs, Nq, 4, device=dev) < torch.tensor([0.05, 0.3, 0.6], device=dev).view(3, 1, 1, 1)
    args = dict(spatial_shapes=torch.tensor(maps, device=dev), level_start_index=torch.tensor([0, 126], device=dev),
                reference_points_cam=torch.rand(cams, bs, Nq, 4, 3, device=dev), bev_mask=mask, value_dpt_dist=dist)
    leaves = [query, feats, dist] + list(layer.parameters())
    got = []
    for pad in (-64.0, 0.0):
        monkeypatch.setattr(spatial_cross_attention, "_OUTSIDE", pad)
        out = layer(query, feats, feats, **args)
        got.append([out.detach()] + list(torch.autograd.grad(out.square().sum(), leaves)))
    for a, b in zip(*got):
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4 * b.abs().max().item())


def test_counting_started_ahead():
    from dfa3D.rebatch import camera_count, camera_index
    g = torch.Generator(device="cuda").manual_seed(2)
    for cams, Nq in ((6, 22500), (1, 1), (3, 1000)):
        hit = torch.rand(cams, Nq, generator=g, device="cuda") < 0.3
        counted = camera_count(hit)
        other = torch.ones(1 << 24, device="cuda").cumsum(0)             # work behind the counting
        index, pos, longest = camera_index(hit, counted)
        want = camera_index(hit)
        assert longest == int(hit.sum(1).max()) == want[2] and torch.equal(index, want[0]) and torch.equal(pos, want[1])
        del other
    assert camera_count(hit.t()) is None and camera_count(hit.float()) is None and camera_count(hit.cpu()) is None


def test_lists_under_a_default_device():
    """A program whose new tensors go to the GPU unless it says otherwise: the counts still come to host memory."""
    from dfa3D.rebatch import camera_index
    hit = torch.rand(6, 500, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda") < 0.3
    want = camera_index(hit)
    with torch.device("cuda"):
        got = camera_index(hit)
    assert got[2] == want[2] and torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("train", [False, True])
def test_layer_with_the_value_side_first(train):
    """Launched before the camera lists, and inside the attention module, as it is where a hook looks on: the same result."""
    from dfa3D.modules import SpatialCrossAttention_DFA3D
    torch.manual_seed(1)
    dev, cams, bs, Nq, E, maps = "cuda", 2, 2, 5000, 64, [(9, 14)]
    layer = SpatialCrossAttention_DFA3D(embed_dims=E, num_cams=cams, bev_h=50, bev_w=100, dropout=0.0, num_head=4,
                                        deformable_attention=dict(embed_dims=E, num_heads=4, num_levels=1, num_points=4)).to(dev)
    for p in layer.parameters():
        torch.nn.init.normal_(p, std=0.1)
    query = torch.randn(bs, Nq, E, device=dev, requires_grad=train)
    feats = torch.randn(cams, 126, bs, E, device=dev)
    args = dict(spatial_shapes=torch.tensor(maps, device=dev), level_start_index=torch.tensor([0], device=dev),
                reference_points_cam=torch.rand(cams, bs, Nq, 4, 3, device=dev), bev_mask=torch.rand(cams, bs, Nq, 4, device=dev) < 0.3,
                value_dpt_dist=torch.rand(cams, 126, bs, 8, device=dev).softmax(-1))
    with torch.set_grad_enabled(train):
        got = layer(query, feats, feats, **args)
        seen = []
        layer.deformable_attention.register_forward_pre_hook(lambda m, a, kw: seen.append(kw.get("value_side")), with_kwargs=True)
        want = layer(query, feats, feats, **args)
        with pytest.raises(ValueError, match="levels"):
            layer(query, feats, feats, **{**args, "spatial_shapes": torch.tensor(maps * 2, device=dev)})
    assert seen == [None] * 2 and torch.equal(got, want)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16], ids=["fp64", "fp32", "bf16"])
def test_scale_has_the_default_dtype(dtype):
    """A program in double precision averages with 1/3 in double precision."""
    from dfa3D.rebatch import camera_hits
    mask = torch.rand(5, 1, 700, 4, generator=torch.Generator().manual_seed(1)) < 0.3
    held = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        hit, scale = camera_hits(mask.cuda())
        want_hit, want_scale = camera_hits(mask)
    finally:
        torch.set_default_dtype(held)
    assert scale.dtype == dtype and torch.equal(hit.cpu(), want_hit) and torch.equal(scale.cpu(), want_scale)
