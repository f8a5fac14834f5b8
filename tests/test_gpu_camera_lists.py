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
