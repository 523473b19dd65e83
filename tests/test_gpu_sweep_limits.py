"""Row sweeps at the limits of their rows (LDS, held chunks, scratch) against
the CPU oracle.  Integer costs: every output bit-exact.  The launches are
counted, so that a form of the aggregation that steps in unseen fails."""
import numpy as np
import pytest

from regard3d_mvs_amd import StereoOptions, synth
from test_gpu_parity import _match_both, gpu  # noqa: F401

pytestmark = pytest.mark.gpu

RAW = dict(speckle_size=0, median=False)
# Launches of a level: path scans, full-range scans, sweeps of one or of three
# paths with two horizontal path scans, and both kinds of sweep with them.
SCANS, FULL, SWEEPS, MIXED = 8, 1, 3, 4


def test_rows_past_a_million_words(gpu):  # noqa: F811
    """Tiles of up to 736 columns whose pixels mostly hold all 4000 labels (the
    coarse level finds little in noise, and nothing fills it): rows of up to
    181754 chunks, past 2^20 words of a scratch row."""
    rng = np.random.default_rng(59)
    left = rng.integers(0, 65536, (24, 4700)).astype(np.uint16)
    right = np.roll(left, -9, 1)
    right[8:16] = rng.integers(0, 65536, (8, 4700))
    g, _ = _match_both(gpu, left, right, None, None, -2000, 4000,
                       StereoOptions(p1=1, p2=2, p2_adapt=0, levels=1, range_radius=0, range_fill=0, uniqueness=0.3,
                                     tile_size=700, **RAW))
    assert g.aggregate_launches < 2 * SCANS


# Rows far below an LDS row: few tiles (one path a sweep) and many (three).
@pytest.mark.parametrize("w,h", [(60, 40), (200, 180)])
def test_narrow_tiles(gpu, w, h):  # noqa: F811
    p = synth.make_pair(w, h, 16, 17)
    g, _ = _match_both(gpu, p.left, p.right, None, None, 0, 16,
                       StereoOptions(levels=1, tile_size=16, tile_margin=2, tile_blend=0))
    assert g.aggregate_launches == FULL + SWEEPS


# 110 tiles of 80 columns, rows of up to 2560 chunks where an LDS row of three
# paths holds 1650.  A patch of noise: 7 tiles whose mean row is past that are
# swept path by path, the others, 5 of them with some such rows, three paths
# at once.  Rows of noise: 34 of the tiles have a few such rows, 21 of them rows of
# more chunks than the threads hold; all are swept three paths at once.
@pytest.mark.parametrize("noise,launches", [("patch", MIXED), ("rows", SWEEPS)])
@pytest.mark.parametrize("p2", [200, 300])
def test_three_path_rows_past_lds(gpu, noise, launches, p2):  # noqa: F811
    p = synth.make_pair(704, 640, 48, 13)
    rng = np.random.default_rng(73)
    right = p.right.copy()
    if noise == "patch":
        right[200:360, 200:480] = rng.integers(0, 65536, (160, 280))
    else:
        for y in (100, 300, 500):
            right[y:y + 10] = rng.integers(0, 65536, (10, 704))
    g, _ = _match_both(gpu, p.left, right, None, None, -256, 512,
                       StereoOptions(levels=1, p2=p2, range_fill=0, range_radius=3 if noise == "patch" else 0,
                                     uniqueness=0.3, tile_size=64, tile_margin=8, tile_blend=0, **RAW))
    assert g.aggregate_launches == (FULL if p2 <= 255 else SCANS) + launches
