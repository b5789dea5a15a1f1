"""The normals view of images that 8 x 8 tiles cover badly (one row, one column, a few of either, just above
a tile), which it takes 64 pixels at a time in order; against the oracle as the others."""
import pytest

from test_gpu_pick_normals import test_normals_and_picks_match_the_oracle as matches_the_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(1, 63), (1, 64), (1, 65), (64, 1), (129, 1), (1, 1000), (1000, 1), (7, 200), (333, 4), (9, 9), (57, 9), (64, 57)])
@pytest.mark.parametrize("lds", [16, 32])
def test_thin_images(W, H, lds):
    matches_the_oracle(W, H, lds)
