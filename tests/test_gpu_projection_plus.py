"""A projection and what is added to it (the residual) in one kernel: equal to the bit to the kernel's product plus the addend, in every kernel that forms
such a product (tile sizes by rows and width; rows around a tile's edge), where sums are odd (infinities, NaN), and through autograd; and the forms that the
kernel does not take."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.view(torch.int32)


@pytest.mark.parametrize("N,O,K", [(1, 64, 64), (63, 256, 256), (65, 130, 100), (5000, 256, 256), (9000, 130, 64), (22500, 256, 256), (22529, 256, 200), (33, 4096, 128)])
def test_product_and_sum_in_one(N, O, K):
    from dfa3D.modules import projection
    torch.manual_seed(N + O)
    x, w, b, r = (torch.randn(s, device="cuda") for s in ((N, K), (O, K), (O,), (N, O)))
    x[N // 2, 3], r[0, 1], r[N - 1, O - 1] = float("inf"), float("nan"), float("-inf")       # an odd sum of the product, and odd addends
    got, want = projection._product(x, w, b, r), projection._product(x, w, b) + r
    odd = want.isnan()
    assert torch.equal(got.isnan(), odd) and torch.equal(_bits(got)[~odd], _bits(want)[~odd])


@pytest.mark.parametrize("N", [50, 7000])
def test_through_autograd(N):
    from dfa3D.modules.projection import Projection, projection_plus
    torch.manual_seed(N)
    layer = Projection(256, 128).cuda()
    x, r = torch.randn(2, N, 256, device="cuda", requires_grad=True), torch.randn(2, N, 128, device="cuda", requires_grad=True)
    leaves, g = (x, r, layer.weight, layer.bias), torch.randn(2, N, 128, device="cuda")
    got, want = projection_plus(layer, x, r), layer(x) + r
    assert "Plus" in got.grad_fn.name() and torch.equal(got, want)
    for a, c in zip(torch.autograd.grad(got, leaves, g), torch.autograd.grad(want, leaves, g)):
        assert torch.equal(a, c)
    # twice: torch operations
    def second(f):
        first, = torch.autograd.grad((f() ** 2).sum(), x, create_graph=True)
        return torch.autograd.grad(first.sum(), (x, layer.weight))
    for a, c in zip(second(lambda: projection_plus(layer, x, r)), second(lambda: layer(x) + r)):
        torch.testing.assert_close(a, c, rtol=1e-4, atol=1e-4 * float(c.abs().max()))
    with torch.no_grad():
        assert torch.equal(projection_plus(layer, x, r), want)


def test_other_forms_are_as_before():
    from dfa3D.modules.projection import Projection, projection_plus
    layer = Projection(64, 64).cuda()
    x, r = torch.randn(3, 40, 64, device="cuda"), torch.randn(3, 40, 64, device="cuda")
    forms = [r[:1], r[..., :1], r.transpose(0, 1).contiguous().transpose(0, 1), r.double(), r.bfloat16(), torch.tensor(2.0), r.clone().requires_grad_()]
    for add in forms:
        for grad in (True, False):
            with torch.set_grad_enabled(grad):
                got, want = projection_plus(layer, x, add), layer(x) + add
            assert got.dtype == want.dtype and torch.equal(got, want) and got.requires_grad == want.requires_grad
    with torch.autocast("cuda", torch.bfloat16):
        got, want = projection_plus(layer, x, r), layer(x) + r
        assert got.dtype == want.dtype and torch.equal(got, want)
    seen = []
    layer.register_forward_hook(lambda *a: seen.append(1))
    projection_plus(layer, x, r)
    assert seen == [1]


@pytest.mark.parametrize("p,train", [(0.0, True), (0.5, False), (0.5, True)])
def test_layer_drops_where_it_is_to(p, train):
    from dfa3D.modules import SpatialCrossAttention_DFA3D
    torch.manual_seed(0)
    layer = SpatialCrossAttention_DFA3D(embed_dims=32, num_cams=1, bev_h=8, bev_w=8, dropout=p, num_head=4,
                                        deformable_attention=dict(embed_dims=32, num_heads=4, num_levels=1, num_points=4)).cuda().train(train)
    query, feats = torch.randn(1, 64, 32, device="cuda"), torch.randn(1, 54, 1, 32, device="cuda")
    got = []
    layer.output_proj.register_forward_hook(lambda m, i, o: got.append(o))      # with a hook the sum is torch's
    args = dict(query_pos=None, spatial_shapes=torch.tensor([(6, 9)], device="cuda"), level_start_index=torch.tensor([0], device="cuda"),
                reference_points_cam=torch.rand(1, 1, 64, 4, 3, device="cuda"), bev_mask=torch.ones(1, 1, 64, 4, dtype=torch.bool, device="cuda"),
                value_dpt_dist=torch.rand(1, 54, 1, 8, device="cuda").softmax(-1))
    hooked = layer(query, feats, feats, **args) - query
    layer.output_proj._forward_hooks.clear()
    bare = layer(query, feats, feats, **args) - query
    if p and train:
        assert 0.4 < (hooked == 0).float().mean() < 0.6 and 0.4 < (bare == 0).float().mean() < 0.6
    else:
        torch.testing.assert_close(bare, hooked, rtol=0, atol=0)
