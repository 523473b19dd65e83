"""combine_pairs at the edges of its register lists (2, 4, 8 and 16 pairs):
bit-exact against the CPU oracle, with noise that makes pairs disagree and the
least-squares fit drop some, maps with and without confidences, non-finite
values, and a grid that leaves the maps' borders."""
import numpy as np
import pytest

from regard3d_mvs_amd.multiview import Rig
from oracle import oracle as O
from regard3d_mvs_amd import MultiStereoOptions, PairGeometry

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(hip_runtime):
    from regard3d_mvs_amd.native import Matcher
    with Matcher(0) as m:
        yield m


@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 8, 9, 15, 16])
def test_pair_counts(gpu, count):
    rng = np.random.default_rng(count)
    angles = np.linspace(0, 2 * np.pi, count, endpoint=False)
    rig = Rig([(0.6 * np.cos(a), 0.6 * np.sin(a), 0.05 * np.cos(3 * a)) for a in angles])
    pairs = []
    for i, c in enumerate(rig.partners):
        p = rig.pair(c, shift=float(rng.choice([0.0, 0.0, 3.0])))
        d = p.disparity + rng.normal(0.0, 0.8, p.disparity.shape).astype(np.float32)
        hole = rng.random(d.shape)
        d[hole < 0.1] = np.inf
        d[hole > 0.98] = np.nan
        conf = None if i % 3 == 1 else rng.random(d.shape).astype(np.float32)
        pairs.append(PairGeometry(p.grid_to_rect, p.fb, p.offset, p.partner_center, d, conf))
    for opt in (MultiStereoOptions(), MultiStereoOptions(inlier_px=3.0, max_reprojection_px=0.5),
                MultiStereoOptions(inlier_px=3.0, max_reprojection_px=1.0, min_angle_deg=6.0, min_pairs=2)):
        for a, b in zip(gpu.combine_pairs(rig.grid(), pairs, opt), O.combine_pairs(rig.grid(), pairs, opt)):
            np.testing.assert_array_equal(np.asarray(a).view(np.uint8), np.asarray(b).view(np.uint8))
