"""Tests of the tile kernels and of the binning before them that go through the Functions with few points, once more with launch options in force: by
size their gradients would come from the direct kernels.  What is named for a path asks for scratch, so that no line drawn elsewhere can empty it."""
import pytest

from dfa3D import _lib
from test_gpu_no_bins import test_gradients_arriving_at_every_output, test_more_tiles_than_counters  # noqa: F401
from test_gpu_parity import (test_bf16_odd_shapes, test_binning_fallbacks, test_cell_kernel_row_lengths_bins_and_tile_edges,  # noqa: F401
                             test_degenerate_level_shapes_and_sixteen_levels, test_every_point_in_one_pixel_cell,
                             test_fp32_one_stage_matches_checker_tiny, test_fp32_random_shapes_match_checker,
                             test_fp32_random_shapes_two_stage_and_shared_distribution, test_gradient_through_depth_score_output,
                             test_more_tiles_than_the_block_histogram_holds, test_non_finite_and_huge_locations_are_skipped,
                             test_non_finite_grad_output_stays_in_the_rows_it_touches, test_plain_deformable_attention_matches_grid_sample,
                             test_shared_distribution_and_weight_update)
from test_gpu_shared_keys import test_bfloat16_gradients, test_float32_gradients  # noqa: F401

pytestmark = pytest.mark.gpu

_NAMED = {"test_more_tiles_than_the_block_histogram_holds", "test_binning_fallbacks", "test_every_point_in_one_pixel_cell",
          "test_non_finite_grad_output_stays_in_the_rows_it_touches", "test_more_tiles_than_counters", "test_gradients_arriving_at_every_output",
          "test_cell_kernel_row_lengths_bins_and_tile_edges", "test_non_finite_and_huge_locations_are_skipped"}
_CODE_AT = {"dfa3d_fused_backward_workspace_bytes": 9, "dfa3d_wms_deform_attn_backward_workspace_bytes": 7,
            "dfa3d_ms_depth_score_sample_backward_workspace_bytes": 7}


@pytest.fixture(autouse=True)
def scratch(request, monkeypatch):
    """The bytes of scratch that the float32 and bfloat16 backwards of a test asked for."""
    lib, sizes = _lib.lib(), []

    def noted(name, at):
        ask = getattr(lib, name)

        def asked(*args):
            size = ask(*args)
            if args[at] in (_lib.DFA3D_F32, _lib.DFA3D_BF16):
                sizes.append(size)
            return size
        return asked

    for name, at in _CODE_AT.items():
        monkeypatch.setattr(lib, name, noted(name, at))
    with _lib.launch_options(chunk=0):
        yield
    if request.node.originalname in _NAMED:
        assert sizes and all(sizes), sizes
