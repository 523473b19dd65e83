"""The three forms of the aggregation (full-range scans, row sweeps, path
scans) against the CPU oracle at the sizes where they change over or run out
of lanes, LDS rows or held chunks.  Integer costs: every output bit-exact."""
import numpy as np
import pytest

from refscenes import Texture, render_pair
from regard3d_mvs_amd import StereoOptions, synth
from test_gpu_parity import _match_both, gpu, same_bits  # noqa: F401

pytestmark = pytest.mark.gpu

RAW = dict(speckle_size=0, median=False)


# Chunks of 16 labels against lanes per scanline: 1, 2, 3, 5, 8, 9, 17, 32 and
# (past the 32 lanes) 33 chunks; images of one pixel, below and past a wave.
@pytest.mark.parametrize("nd", [16, 32, 48, 80, 128, 144, 272, 512, 528])
def test_full_range_labels(gpu, nd):  # noqa: F811
    left, right, _ = render_pair(Texture(31), 67, 35, lambda x, y: 4.0 + 0.1 * x - 0.05 * y)
    _match_both(gpu, left, right, None, None, -3, nd, StereoOptions(levels=0, **RAW))


@pytest.mark.parametrize("shape", [(1, 1), (1, 40), (40, 1), (64, 64), (65, 130)])
def test_full_range_shapes(gpu, shape):  # noqa: F811
    rng = np.random.default_rng(shape[0])
    left = rng.integers(0, 65536, shape).astype(np.uint16)
    right = rng.integers(0, 65536, shape).astype(np.uint16)
    _match_both(gpu, left, right, None, None, -8, 32, StereoOptions(levels=0, tile_size=64, tile_margin=4, **RAW))


# The largest P2 whose path costs fit bytes, the next, and the largest allowed
# (path costs of 14 bits, sums that wrap at 16).
@pytest.mark.parametrize("p2", [255, 256, 8000])
@pytest.mark.parametrize("levels", [0, 1])
def test_penalties(gpu, p2, levels):  # noqa: F811
    left, right, _ = render_pair(Texture(37), 150, 70, lambda x, y: np.where(x < 60, 6.0, 17.5) + 0.03 * y)
    _match_both(gpu, left, right, None, None, 0, 64,
                StereoOptions(p1=min(p2, 1000) // 8, p2=p2, p2_adapt=0, levels=levels, **RAW))


# Rows of a tile against the sweeps' limits: one column; 1000 columns of at
# least 144 labels (9000 chunks: past the LDS rows and the held chunks, in
# scratch); 1100 columns (past a block's threads: path scans).
@pytest.mark.parametrize("w,margin,tile", [(1, 4, 512), (1000, 64, 1024), (1100, 4, 2048)])
def test_sweep_rows(gpu, w, margin, tile):  # noqa: F811
    left, right, _ = render_pair(Texture(41), w, 24, lambda x, y: 30.0 + 0.02 * x + 0.3 * y)
    _match_both(gpu, left, right, None, None, 0, 256,
                StereoOptions(levels=1, range_margin=margin, tile_size=tile, **RAW))


# Many small tiles (three paths per sweep) and few (one path), with edges.
@pytest.mark.parametrize("tile", [24, 512])
def test_sweep_tiles(gpu, tile):  # noqa: F811
    p = synth.make_pair(301, 199, 48, 7)
    _match_both(gpu, p.left, p.right, None, None, 0, 48, StereoOptions(levels=1, tile_size=tile, tile_margin=9, tile_blend=6))


def test_small_budget_scans(hip_runtime, gpu):  # noqa: F811
    """Where the memory left holds neither planes nor slices, path scans give
    the same maps."""
    from regard3d_mvs_amd.native import Matcher
    p = synth.make_pair(640, 480, 64, 5)
    for levels in (0, 1):
        o = StereoOptions(levels=levels)
        ref = gpu.match(p.left, p.right, dmin=0, nd=64, options=o, debug=True)
        with Matcher(0, hbm_budget=160 << 20) as small:
            got = small.match(p.left, p.right, dmin=0, nd=64, options=o, debug=True)
        assert got.aggregate_launches > ref.aggregate_launches
        for k in ("disparity", "confidence", "labels", "lr_mask"):
            same_bits(getattr(got, k), getattr(ref, k))


# Enough scanlines that a lane takes eight labels also where D is small
# (16 labels: 4 lanes of four, 24576 scanlines at 256 CUs).
@pytest.mark.parametrize("nd", [16, 32, 48, 128])
def test_full_range_many_scanlines(gpu, nd):  # noqa: F811
    left, right, _ = render_pair(Texture(43), 2600, 21, lambda x, y: 5.0 + 0.002 * x + 0.1 * y)
    _match_both(gpu, left, right, None, None, 0, nd, StereoOptions(levels=0, **RAW))


def test_sweep_few_wide_rows(gpu):  # noqa: F811
    """Rows of far more chunks than a thread holds two of, in tiles whose mean
    row has fewer than one per thread: noise in a few rows widens their ranges."""
    left, right, _ = render_pair(Texture(47), 480, 400, lambda x, y: 60.0 + 0.02 * x + 0.01 * y)
    rng = np.random.default_rng(47)
    right = right.copy()
    right[200:206] = rng.integers(0, 65536, right[200:206].shape)
    _match_both(gpu, left, right, None, None, 0, 256, StereoOptions(levels=1, range_margin=4, **RAW))


# One tile of more columns than 16 bits count: full-range scans, path scans
# with label ranges, and penalties past a byte.
@pytest.mark.parametrize("levels,p2", [(0, 100), (1, 100), (0, 300)])
def test_tile_of_70000_columns(gpu, levels, p2):  # noqa: F811
    rng = np.random.default_rng(53)
    left = rng.integers(0, 65536, (24, 70000)).astype(np.uint16)
    right = np.roll(left, -9, 1)
    _match_both(gpu, left, right, None, None, 0, 32,
                StereoOptions(levels=levels, p1=10, p2=p2, tile_size=100000, tile_margin=4, **RAW))
