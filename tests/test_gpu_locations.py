"""Sampling locations in one kernel against the module's tensor operations: row and point counts around the blocks, every
ratio of points to anchors, gradients, and the calls that keep the tensor operations."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _plain(mod, query, ref, shapes):
    bs, Q, _ = query.shape
    M, L, P, Z = mod.num_heads, mod.num_levels, mod.num_points, ref.shape[2]
    uv = mod.sampling_offsets(query).view(bs, Q, M, L, P, 2)
    dz = mod.sampling_offsets_depth(query).view(bs, Q, M, L, P, 1)
    off = torch.cat([uv, dz], -1) / shapes[:, [1, 0, 2]].to(query.dtype)[None, None, None, :, None, :]
    return (off.view(bs, Q, M, L, P // Z, Z, 3) + ref[:, :, None, None, None]).view(bs, Q, M, L, P, 3)


@pytest.mark.parametrize("bs,Q,M,L,P,Z", [(1, 1, 1, 1, 1, 1), (2, 17, 8, 4, 8, 4), (6, 300, 8, 1, 8, 2), (1, 33, 3, 3, 5, 5),
                                          (3, 15, 2, 2, 6, 3), (1, 16, 8, 4, 10, 1), (1, 0, 4, 2, 4, 4)])
def test_locations_and_gradients(bs, Q, M, L, P, Z):
    from dfa3D.modules import MSDeformableAttention3D_DFA3D
    torch.manual_seed(Q)
    dev = torch.device("cuda:0")
    mod = MSDeformableAttention3D_DFA3D(embed_dims=8 * M, num_heads=M, num_levels=L, num_points=P).to(dev)
    torch.nn.init.normal_(mod.sampling_offsets.weight)
    torch.nn.init.normal_(mod.sampling_offsets_depth.weight)
    query = torch.randn(bs, Q, 8 * M, device=dev, requires_grad=True)
    ref = torch.rand(bs, Q, Z, 3, device=dev)
    shapes = torch.tensor([[29 - 3 * l, 50 - 7 * l, 64] for l in range(L)], device=dev)
    got, want = mod.sampling_locations(query, ref, shapes), _plain(mod, query, ref, shapes)
    assert torch.equal(got, want)                              # the same roundings
    leaves = [query, mod.sampling_offsets.weight, mod.sampling_offsets_depth.bias]
    g = torch.randn_like(want)
    for a, b in zip(torch.autograd.grad(got, leaves, g, retain_graph=True), torch.autograd.grad(want, leaves, g)):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)
    # a gradient that is recorded, reference points that want one, other layouts and types: tensor operations
    first = torch.autograd.grad((got ** 3).sum(), [query], create_graph=True)[0]
    if Q:
        assert torch.autograd.grad(first.sum(), [query])[0].abs().max() > 0
        many = torch.randn(2, *got.shape, device=dev)
        batch, = torch.autograd.grad(mod.sampling_locations(query, ref, shapes), [mod.sampling_offsets_depth.bias], many, is_grads_batched=True)
        plain, = torch.autograd.grad(_plain(mod, query, ref, shapes), [mod.sampling_offsets_depth.bias], many, is_grads_batched=True)
        torch.testing.assert_close(batch, plain, rtol=1e-4, atol=1e-4)
    wanting = ref.clone().requires_grad_()
    moved = mod.sampling_locations(query, wanting, shapes)
    assert torch.equal(moved, want) and torch.autograd.grad(moved.sum(), [wanting])[0].shape == ref.shape
    strided = torch.rand(bs, Z, Q, 3, device=dev).transpose(1, 2)
    assert torch.equal(mod.sampling_locations(query, strided, shapes), _plain(mod, query, strided, shapes))
    with torch.no_grad():
        assert torch.equal(mod.sampling_locations(query, ref, shapes), want)
    double = mod.double()
    assert torch.equal(double.sampling_locations(query.double(), ref.double(), shapes), _plain(double, query.double(), ref.double(), shapes))
