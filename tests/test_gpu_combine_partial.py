"""combine_pairs with maps that cover parts of the grid, so that waves see some
of the pairs only, or none; bit-exact against the CPU oracle."""
import numpy as np
import pytest

from regard3d_mvs_amd.multiview import Rig
from oracle import oracle as O
from regard3d_mvs_amd import MultiStereoOptions, PairGeometry
from test_gpu_combine_counts import gpu  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 2, 4, 7, 16])
def test_partly_seen_grids(gpu, count):  # noqa: F811
    rng = np.random.default_rng(count)
    angles = np.linspace(0, 2 * np.pi, count, endpoint=False)
    rig = Rig([(0.6 * np.cos(a), 0.6 * np.sin(a), 0.0) for a in angles])
    pairs = []
    for i, c in enumerate(rig.partners):
        p = rig.pair(c)
        h, w = p.disparity.shape
        h, w = ((h, w), (h // 3, w), (h, w // 5), (1, 1))[i % 4]
        d = np.ascontiguousarray(p.disparity[:h, :w])
        conf = None if i % 3 == 1 else rng.random(d.shape).astype(np.float32)
        pairs.append(PairGeometry(p.grid_to_rect, p.fb, p.offset, p.partner_center, d, conf))
    for opt in (MultiStereoOptions(), MultiStereoOptions(min_pairs=2)):
        for a, b in zip(gpu.combine_pairs(rig.grid(), pairs, opt), O.combine_pairs(rig.grid(), pairs, opt)):
            np.testing.assert_array_equal(np.asarray(a).view(np.uint8), np.asarray(b).view(np.uint8))
