"""The local operator's sweeps once more with the gradient kernels of the larger layers: the layers of the suite are small, so
that the oracle is quick, and most of their gradients come from the one-launch form by default (dk_local_small.hip)."""
import pytest

from test_gpu_local import (  # noqa: F401  (collected again here)
    test_bf16_group_of_one_channel_keeps_fp32_matrix_instructions,
    test_filter_gradient_with_two_slices_of_cells_per_launch,
    test_fp32_matches_oracle,
    test_grad_rotation_by_channel_pairs_on_bfloat16_tensors,
    test_half_precisions_match_fp32_oracle,
    test_non_contiguous_inputs_and_needs_input_grad_gating,
    test_rotation_clip_inside_the_operator,
    test_taps_outside_the_scope_and_nan_free_borders,
)
from test_gpu_graph import test_local_operator_forward_and_backward_replay_from_a_graph  # noqa: F401
from test_gpu_nhwc import (  # noqa: F401
    test_equals_the_planar_operator_on_the_same_tensors,
    test_fp32_matches_oracle as test_channels_last_fp32_matches_oracle,
    test_half_precision_filter_gradient_at_stride_2_keeps_float32_where_the_pixels_cancel,
    test_half_precisions_match_fp32_oracle as test_channels_last_half_precisions_match_fp32_oracle,
    test_quads_at_stride_2_and_eight_channels_per_lane,
)
from test_gpu_random_shapes import (  # noqa: F401
    test_local_operator_on_random_geometries,
    test_local_operator_on_random_geometries_in_16_bits,
)

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _larger_kernels(switch_off):
    switch_off("DK_NO_SMALL_BACKWARD")
