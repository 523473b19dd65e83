"""Tile rows of several strips (2^16 columns each): path scans, costs and
selection against the CPU oracle.  Integer costs: every output bit-exact."""
import numpy as np
import pytest

from regard3d_mvs_amd import StereoOptions
from test_gpu_parity import _match_both, gpu  # noqa: F401

pytestmark = pytest.mark.gpu

WIDE = dict(speckle_size=0, median=False, tile_size=1 << 20, tile_margin=4, memory_budget=1 << 42)


def _pair(w, h, shift, seed):
    left = np.random.default_rng(seed).integers(0, 65536, (h, w)).astype(np.uint16)
    return left, np.roll(left, -shift, 1)


def test_row_of_2_to_28_cells(gpu):  # noqa: F811
    """70000 columns of 4000 labels: more chunks in a row than 24 bits count."""
    left, right = _pair(70000, 2, 9, 71)
    g, _ = _match_both(gpu, left, right, None, None, -2000, 4000, StereoOptions(levels=0, **WIDE))
    assert g.cells >= 2 * 2 ** 28


# The last column of a strip, the first of the next, and three strips; label
# ranges, and one level by path scans.
@pytest.mark.parametrize("w", [65535, 65536, 65537, 140001])
@pytest.mark.parametrize("levels,p2", [(1, 200), (0, 300)])
def test_strips(gpu, w, levels, p2):  # noqa: F811
    left, right = _pair(w, 12, 6, w)
    _match_both(gpu, left, right, None, None, 0, 32,
                StereoOptions(levels=levels, p1=10, p2=p2, p2_adapt=0, range_margin=2, **WIDE))
