"""Speckle removal at the edges of its 32 x 32 blocks, bit-exact against the CPU
oracle: maps of one pixel to just past two blocks, steps that join nothing,
neighbours or (infinite) everything but NaN, segments at and around min_size.
The GPU gives removed and NaN pixels alike +inf; the oracle leaves NaN."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(hip_runtime):
    from regard3d_mvs_amd.native import Matcher
    with Matcher(0) as m:
        yield m


@pytest.mark.parametrize("h,w", [(1, 1), (1, 65), (33, 1), (31, 32), (32, 33), (64, 64), (65, 97), (300, 31)])
@pytest.mark.parametrize("max_diff", [0.0, 0.6, np.inf])
def test_block_edges(gpu, h, w, max_diff):
    rng = np.random.default_rng(h * 131 + w)
    d = np.round(rng.random((h, w)) * 2.0).astype(np.float32) * 0.5
    d[rng.random(d.shape) < 0.1] = np.inf
    d[rng.random(d.shape) < 0.03] = np.nan
    for size in (2, 3, 33, h * w // 2 + 1, h * w, h * w + 1):
        a, b = gpu.remove_speckles(d, size, max_diff), O.remove_speckles(d, size, max_diff)
        b = np.where(np.isnan(b), np.float32(np.inf), b)
        np.testing.assert_array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))
