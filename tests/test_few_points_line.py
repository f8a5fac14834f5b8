"""Where the line between the direct and the tile kernels of a backward lies, asked on the host: by the scratch that a call wants.  On both sides of each
term of the rule: atomics against tiles, points that may lie close together, float sums of bfloat16 gradients."""
import ctypes

import pytest

from dfa3D import _lib


def _direct(kind, B, S, L, Q, P, C=32, D=64, M=8, heads=8, code=_lib.DFA3D_F32):
    lib, ask = _lib.lib(), []
    for direct in (_lib.DFA3D_FEW_POINTS, 0):
        o = ctypes.pointer(_lib.LaunchOptions(direct=direct))
        if kind == "fused":
            ask.append(lib.dfa3d_fused_backward_workspace_bytes(B, S, M, C, D, L, Q, P, heads, code, o))
        elif kind == "plain":
            ask.append(lib.dfa3d_wms_deform_attn_backward_workspace_bytes(B, S, M, C, L, Q, P, code, o))
        else:
            ask.append(lib.dfa3d_ms_depth_score_sample_backward_workspace_bytes(B, S, M, D, L, Q, P, code, o))
    assert ask[1] > 0
    return ask[0] != ask[1]


@pytest.mark.parametrize("kind,B,S,L,P,last,options", [
    ("fused", 2, 3000, 2, 8, 184, {}), ("fused", 2, 3000, 2, 8, 208, dict(heads=1)), ("fused", 2, 3000, 2, 8, 116, dict(C=64)),
    ("fused", 2, 30825, 4, 8, 376, {}), ("fused", 6, 30825, 4, 8, 184, {}), ("fused", 6, 30825, 4, 8, 361, dict(heads=1)),
    ("plain", 2, 2400, 1, 4, 991, {}), ("plain", 6, 30825, 4, 8, 268, {}),
    ("stage 1", 2, 3000, 4, 2, 1543, {}), ("stage 1", 6, 30825, 4, 8, 82, {})])
def test_last_call_of_the_direct_kernels(kind, B, S, L, P, last, options):
    """A point has an atomic per 64 bytes of its four rows and four for its bins, 0.05 ns each; a call has its base and its rows.  The first:
    (19 us + 48000 rows * 0.196 ns) / (256 points a query * 12 * 0.05 ns) = 184.9."""
    assert _direct(kind, B, S, L, last, P, **options) and not _direct(kind, B, S, L, last + 1, P, **options)


@pytest.mark.parametrize("kind,B,S,L,P,last,options", [
    ("plain", 2, 40000, 1, 4, 2000, {}), ("fused", 2, 23200, 1, 8, 1000, dict(D=128)), ("stage 1", 2, 23200, 1, 8, 500, dict(D=112)),
    ("plain", 1, 315, 1, 4, 787, {}), ("fused", 3, 1040, 4, 4, 24, dict(D=16, heads=1))])
def test_points_that_may_lie_close_together(kind, B, S, L, P, last, options):
    """8000 points of a batch element, head and level (4000), ten of a row (2520 rows, 32 points a query), three of a line (3120 lines, 384)."""
    assert _direct(kind, B, S, L, last, P, **options) and not _direct(kind, B, S, L, last + 1, P, **options)


def test_float_sums_of_bfloat16_gradients():
    """384 bytes a row: 80 MB are 208 333 rows.  Rows of 16 channels have float sums from either kind of kernels."""
    b16 = _lib.DFA3D_BF16G
    assert _direct("fused", 1, 26041, 4, 1, 8, code=b16) and not _direct("fused", 1, 26042, 4, 1, 8, code=b16)
    assert _direct("fused", 1, 26042, 4, 1, 8) and _direct("fused", 6, 30825, 4, 1, 8, heads=1, code=b16)
    assert _direct("fused", 6, 30825, 4, 100, 8, C=16, code=b16)
    assert _direct("fused", 2, 3000, 2, 40, 8, code=b16) and not _direct("fused", 2, 3000, 2, 154, 8, code=b16)
