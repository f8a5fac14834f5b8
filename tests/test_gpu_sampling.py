"""Sampling locations and attention weights in one kernel: locations as by their own kernel to the bit, weights and gradients against float64, at every number of
points that lanes share, rows and heads around a workgroup's; logits that are large, equal, infinite and none; and the calls that keep torch's softmax."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


@pytest.mark.parametrize("bs,Q,M,L,P,Z", [(1, 1, 1, 1, 1, 1), (2, 17, 8, 4, 8, 4), (6, 300, 8, 1, 8, 2), (1, 33, 3, 2, 8, 4), (1, 37, 6, 4, 16, 4), (3, 15, 5, 2, 2, 1),
                                          (1, 16, 40, 1, 2, 1), (1, 19, 1, 1, 2, 2), (2, 0, 4, 2, 4, 4)])
def test_against_float64(bs, Q, M, L, P, Z):
    from dfa3D.modules.ms_deform_attn_3d import _LocationsFunction, _SamplingFunction
    torch.manual_seed(Q)
    dev = "cuda"
    uv, dz, logits = (torch.randn(bs, Q, M, L, P, *s, device=dev) for s in ((2,), (1,), ()))
    logits *= 10
    if Q > 2:
        logits[0, 0, 0], logits[0, 1, 0] = 1e30, -3e38
        logits[0, 2, 0, 0, 0] = float("-inf")
    ref, shapes = torch.rand(bs, Q, Z, 3, device=dev), torch.tensor([[29 - 3 * l, 50 - 7 * l, 64] for l in range(L)], device=dev)
    leaves = [t.requires_grad_() for t in (uv, dz, logits)]
    loc, attn = _SamplingFunction.apply(*leaves, ref, shapes)
    alone = _LocationsFunction.apply(uv, dz, ref, shapes)
    assert torch.equal(loc, alone) and loc.requires_grad and attn.requires_grad
    exact = logits.detach().double().flatten(-2).requires_grad_()
    want = exact.softmax(-1)
    # the exponential of a rounded difference, its rounding, a sum of at most 64 and a division: 2 + 10 |x - max| would be safe as well; a few parts in 2^24
    spread = (exact.max(-1, keepdim=True)[0] - exact).detach().clamp(max=104) if Q else exact.detach()
    bound = (8 + spread) * EPS * want.detach() + 1e-37
    ok = want.isfinite()
    assert ((attn.detach().flatten(-2).double() - want.detach()).abs() <= bound)[ok].all() and torch.equal(attn.detach().flatten(-2).isfinite(), ok)
    g, ga = torch.randn_like(loc), torch.randn_like(attn)
    got = torch.autograd.grad((loc, attn), leaves, (g, ga), retain_graph=True)
    locs = torch.autograd.grad(alone, (uv, dz), g)
    assert torch.equal(got[0], locs[0]) and torch.equal(got[1], locs[1])
    want_logits, = torch.autograd.grad(want, exact, ga.double().flatten(-2))
    size = (want.detach() * ga.double().flatten(-2).abs()).sum(-1, keepdim=True) + ga.double().flatten(-2).abs() if Q else 1
    assert ((got[2].flatten(-2).double() - want_logits).abs() <= (12 + 2 * 104) * EPS * want.detach() * size + 1e-36)[ok].all()
    if not Q:
        return
    # recorded gradients, and a gradient of one result alone
    first, = torch.autograd.grad(attn[0, 3:].square().sum(), logits, create_graph=True)
    second, = torch.autograd.grad(first.sum() + (first ** 2).sum(), logits, retain_graph=True) if Q > 3 else (None,)
    if Q > 3:
        e = logits.detach()[0, 3:].double().flatten(-2).requires_grad_()
        f, = torch.autograd.grad(e.softmax(-1).square().sum(), e, create_graph=True)
        s, = torch.autograd.grad(f.sum() + (f ** 2).sum(), e)
        torch.testing.assert_close(second[0, 3:].flatten(-2).double(), s, rtol=1e-4, atol=1e-5)
    only, = torch.autograd.grad(loc.sum(), uv, retain_graph=True)
    torch.testing.assert_close(only, torch.autograd.grad(_LocationsFunction.apply(uv, dz, ref, shapes).sum(), uv)[0], rtol=0, atol=0)


@pytest.mark.parametrize("L,P,kernel", [(4, 8, True), (3, 4, False), (4, 32, False), (1, 1, True)])
def test_module_takes_it_where_it_may(L, P, kernel):
    from dfa3D.modules import MSDeformableAttention3D_DFA3D
    torch.manual_seed(L)
    mod = MSDeformableAttention3D_DFA3D(embed_dims=32, num_heads=4, num_levels=L, num_points=P).cuda()
    uv, dz, logits = (torch.randn(2, 9, 4 * L * P * k, device="cuda", requires_grad=True) for k in (2, 1, 1))
    ref, shapes = torch.rand(2, 9, 1, 3, device="cuda"), torch.tensor([[20, 30, 8]] * L, device="cuda")
    forms = {"plain": (logits, ref, kernel), "strided": (logits.detach().transpose(0, 1).contiguous().transpose(0, 1), ref, False),
             "points": (logits, ref.clone().requires_grad_(), False)}
    for how, (x, r, by_kernel) in forms.items():
        loc, attn = mod._sampling(uv, dz, x, r, shapes, torch.float32)
        assert ("Sampling" in attn.grad_fn.name() if attn.requires_grad else False) == by_kernel, how
        torch.testing.assert_close(attn.flatten(-2), x.view(2, 9, 4, L * P).softmax(-1), rtol=1e-5, atol=1e-7)
        assert torch.equal(loc, mod._locations(uv, dz, r, shapes, torch.float32))
    with torch.autocast("cuda", torch.bfloat16):
        loc, attn = mod._sampling(uv, dz, logits, ref, shapes, torch.float32)
        assert "Sampling" not in attn.grad_fn.name()


def test_with_saved_tensors_elsewhere():
    """Hooks that keep saved tensors on the host, or bring them back as others: the gradients stay the same."""
    from dfa3D.modules.ms_deform_attn_3d import _LocationsFunction, _SamplingFunction
    torch.manual_seed(0)
    uv, dz, logits = (torch.randn(1, 9, 2, 2, 4, *s, device="cuda", requires_grad=True) for s in ((2,), (1,), ()))
    ref, shapes = torch.rand(1, 9, 1, 3, device="cuda"), torch.tensor([[20, 30, 8], [10, 15, 8]], device="cuda")
    want = torch.autograd.grad([t.square().sum() for t in _SamplingFunction.apply(uv, dz, logits, ref, shapes)], (uv, dz, logits))
    # back on the GPU; left on the host (the level table alone: what meets the gradients has to be where they are); strided
    for unpack in (lambda t: t.cuda(), lambda t: t if t.dtype == torch.int64 else t.cuda(), lambda t: t.cuda().t().contiguous().t() if t.dim() == 2 else t.cuda()):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), unpack):
            loc, attn = _SamplingFunction.apply(uv, dz, logits, ref, shapes)
            alone = _LocationsFunction.apply(uv, dz, ref, shapes)
        g = 2 * loc.detach(), 2 * attn.detach()
        for a, b in zip(torch.autograd.grad((loc, attn), (uv, dz, logits), g), want):
            torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-6)
        for a, b in zip(torch.autograd.grad(alone, (uv, dz), g[0]), want):
            torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-6)
