"""The launch option `direct` asked on the host: every value that says yes means always, one value means by size."""
import ctypes

import pytest

from dfa3D import _lib


@pytest.mark.parametrize("direct", [1, 2, 3, -1, -2, 255, 2 ** 31 - 1, -2 ** 31])
def test_any_yes_is_always(direct):
    L, o = _lib.lib(), ctypes.pointer(_lib.LaunchOptions(direct=direct))
    few, many = 100, 40000
    for Q in (few, many):
        assert L.dfa3d_fused_backward_workspace_bytes(6, 30825, 8, 32, 64, 4, Q, 8, 8, _lib.DFA3D_F32, o) == 0
        assert L.dfa3d_fused_backward_workspace_bytes(6, 30825, 8, 32, 64, 4, Q, 8, 8, _lib.DFA3D_BF16G, o) == 0
        assert L.dfa3d_wms_deform_attn_backward_workspace_bytes(6, 30825, 8, 32, 4, Q, 8, _lib.DFA3D_F32, o) == 0
        assert L.dfa3d_ms_depth_score_sample_backward_workspace_bytes(6, 30825, 8, 64, 4, Q, 8, _lib.DFA3D_F32, o) == 0


def test_by_size():
    L = _lib.lib()
    ask = lambda Q, direct: L.dfa3d_fused_backward_workspace_bytes(6, 30825, 8, 32, 64, 4, Q, 8, 8, _lib.DFA3D_F32,
                                                                   ctypes.pointer(_lib.LaunchOptions(direct=direct)))
    assert ask(4, _lib.DFA3D_FEW_POINTS) == 0 < ask(4, 0) and ask(40000, _lib.DFA3D_FEW_POINTS) == ask(40000, 0) > 0
