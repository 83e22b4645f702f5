"""The recurrences for hidden sizes past 256 (four rows and 32 units per
workgroup, W_hh in registers) against the float64 oracle at the edges of their
tiles, and their behaviour when a wait gives up."""
import pytest

from test_gpu_parity import _check_abort_path, _check_layer_against_oracle

pytestmark = pytest.mark.gpu

# forward k ranges of 24, 32, 40 and 48 values per lane (H to 384, 512, 640,
# 768) and backward tiles of 2 and 3 per wavefront (H to 512, 768), each at its
# first and last H; slices and rows partly empty; scalar weight loads (H not a
# multiple of 4); several launches over batch slices, the last one shorter
WIDE_SHAPES = [(1, 3, 5, 257), (4, 1, 4, 384), (3, 4, 3, 385), (5, 2, 8, 512), (6, 3, 7, 513), (2, 4, 4, 640),
               (9, 2, 2, 641), (7, 3, 4, 767), (4, 3, 8, 768), (131, 3, 4, 500), (70, 2, 3, 660)]


@pytest.mark.parametrize("B,T,I,H", WIDE_SHAPES)
def test_wide_layer_matches_oracle(gpu, oracle, B, T, I, H):
    _check_layer_against_oracle(gpu, oracle, "auto", B, T, I, H)


@pytest.mark.parametrize("B,T,H", [(5, 12, 512), (70, 6, 700)])
def test_wide_timed_out_waits_abort_with_nan(gpu, oracle, hip_lib, B, T, H):
    _check_abort_path(gpu, oracle, hip_lib, "auto", B, T, H)
