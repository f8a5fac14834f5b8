"""Weight and bias gradients of several layers on the same rows in one pair of launches: equal to the bit to those of each layer alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 255, 257, 4097, 30001])
@pytest.mark.parametrize("K,widths,bias", [(256, (512, 256, 256), (True, True, True)), (64, (2, 130, 128, 258), (True, False, True, False)),
                                           (300, (64, 64), (False, True)), (4, (2048,), (True,))])
def test_each_layer_as_alone(N, K, widths, bias):
    from dfa3D.modules import projection
    torch.manual_seed(N + K)
    x, grads = torch.randn(N, K, device="cuda"), [torch.randn(N, O, device="cuda") for O in widths]
    grads[-1][N // 2] = float("inf")                      # sums that are formed again
    got = projection._several_weight_gradients(x, grads, bias)
    for g, want_bias, (weight, b) in zip(grads, bias, got):
        alone, alone_bias = projection._weight_gradients(x, g, want_bias)
        assert torch.equal(weight.view(torch.int32), alone.view(torch.int32)) and (b is None) == (not want_bias)
        assert b is None or torch.equal(b.view(torch.int32), alone_bias.view(torch.int32))


@pytest.mark.parametrize("frozen", [(), (0,), (1, 2), (0, 1, 2)])
def test_with_layers_that_are_not_trained(frozen):
    from dfa3D.modules.projection import Projection, projections
    torch.manual_seed(1)
    layers = [Projection(64, O).cuda() for O in (64, 32, 32)]
    for i in frozen:
        layers[i].bias.requires_grad_(False)
    x = torch.randn(2, 500, 64, device="cuda", requires_grad=True)
    gs = [torch.randn(2, 500, l.out_features, device="cuda") for l in layers]
    for used in ((0, 1, 2), (2,), (0, 2)):                # of whose results a gradient comes back
        outs = projections(x, layers)
        leaves = [x] + [p for i in used for p in layers[i].parameters() if p.requires_grad]
        got = torch.autograd.grad([outs[i] for i in used], leaves, [gs[i] for i in used])
        want = torch.autograd.grad([torch.nn.functional.linear(x, layers[i].weight, layers[i].bias) for i in used], leaves, [gs[i] for i in used])
        for a, c in zip(got, want):
            torch.testing.assert_close(a, c, rtol=1e-4, atol=1e-4 * float(c.abs().max()))


def test_keys_that_the_module_does_not_read():
    from dfa3D.modules import SpatialCrossAttention_DFA3D
    torch.manual_seed(0)
    cams, bs, E = 2, 2, 32
    layer = SpatialCrossAttention_DFA3D(embed_dims=E, num_cams=cams, bev_h=8, bev_w=8, dropout=0.0, num_head=4,
                                        deformable_attention=dict(embed_dims=E, num_heads=4, num_levels=1, num_points=4)).cuda()
    query, feats = torch.randn(bs, 64, E, device="cuda"), torch.randn(cams, 54, bs, E, device="cuda")
    args = dict(spatial_shapes=torch.tensor([(6, 9)], device="cuda"), level_start_index=torch.tensor([0], device="cuda"),
                reference_points_cam=torch.rand(cams, bs, 64, 4, 3, device="cuda"), bev_mask=torch.rand(cams, bs, 64, 4, device="cuda") < 0.2,
                value_dpt_dist=torch.rand(cams, 54, bs, 8, device="cuda").softmax(-1))
    want = layer(query, feats, feats, **args)
    assert torch.equal(layer(query, torch.full_like(feats, float("nan")), feats, **args), want)
    seen = []
    handle = layer.deformable_attention.register_forward_pre_hook(lambda m, a, k: seen.append(k["key"]), with_kwargs=True)
    assert torch.equal(layer(query, feats, feats, **args), want)
    handle.remove()
    assert torch.equal(seen[0], feats.permute(2, 0, 1, 3).reshape(bs * cams, 54, E))
    for bad in (feats[..., :16], feats[:, :, :1], feats[0]):
        with pytest.raises((RuntimeError, ValueError, IndexError)):
            layer(query, bad, feats, **args)
