"""Entry points of the C interface, or forms of their arguments, that the package itself has no use for."""
import pytest
import torch

from dfa3D import _lib

pytestmark = pytest.mark.gpu


def _stream():
    return torch.cuda.current_stream().cuda_stream


def test_lists_without_totals():
    g = torch.Generator().manual_seed(0)
    hit = (torch.rand(3, 2500, generator=g) < 0.3).cuda()
    longest, p = int(hit.sum(1).max()), _lib.ptr
    got = []
    for totals in (None, torch.full((3,), -7, dtype=torch.int32, device="cuda")):
        index, pos = (torch.full((3, n), 99, dtype=torch.int32, device="cuda") for n in (longest, 2500))
        _lib.check(_lib.lib().dfa3d_camera_index(p(hit), p(totals), p(index), p(pos), 3, 2500, longest, _stream()), "dfa3d_camera_index")
        got.append((index, pos))
    for index, pos in got:
        for cam in range(3):
            seen = hit[cam].nonzero()[:, 0].int()
            assert torch.equal(index[cam, :len(seen)], seen) and (index[cam, len(seen):] == -1).all()
            assert torch.equal(pos[cam][hit[cam]], torch.arange(len(seen), dtype=torch.int32, device="cuda")) and (pos[cam][~hit[cam]] == -1).all()
