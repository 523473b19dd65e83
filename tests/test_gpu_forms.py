"""Which form of the aggregation a level takes (full-range scans: one launch;
row sweeps and horizontal path scans: 3, with both kinds of sweep 4; path
scans: 8), by the launches counted, and its maps against the CPU oracle.
Integer costs: every output bit-exact."""
import numpy as np
import pytest

from refscenes import Texture, render_pair
from regard3d_mvs_amd import StereoOptions, synth
from test_gpu_parity import _match_both, gpu, same_bits  # noqa: F401

pytestmark = pytest.mark.gpu

RAW = dict(speckle_size=0, median=False)
FULL, SWEEPS, SCANS = 1, 3, 8


# One full-range level: the last label count and P2 of the full-range scans,
# and the first ones past them.
@pytest.mark.parametrize("nd,p2,launches", [(512, 255, FULL), (528, 255, SCANS), (64, 256, SCANS), (1040, 300, SCANS)])
def test_full_range_form(gpu, nd, p2, launches):  # noqa: F811
    left, right, _ = render_pair(Texture(61), 83, 41, lambda x, y: 4.0 + 0.1 * x - 0.05 * y)
    g, _ = _match_both(gpu, left, right, None, None, -5, nd, StereoOptions(levels=0, p2=p2, p2_adapt=0, **RAW))
    assert g.aggregate_launches == launches


# Device budgets that hold S and the costs of a range (3 bytes per cell) beside
# the pair's images and maps and little more: the chunk map takes the costs'
# place after the path scans, few waves scan at once, and cached blocks of other
# ranges do not end up under smaller volumes.
@pytest.mark.parametrize("w,h,mib", [(1024, 768, 137), (2000, 1500, 303), (2000, 1500, 653)])
def test_tight_budgets(hip_runtime, gpu, w, h, mib):  # noqa: F811
    import torch
    from regard3d_mvs_amd.native import Matcher
    rng = np.random.default_rng(w)
    left = rng.integers(0, 65536, (h, w)).astype(np.uint16)
    images = [torch.from_numpy(a).cuda() for a in (left, np.roll(left, -21, 1))]
    o = StereoOptions(levels=0, **RAW)
    ref = gpu.match(*images, dmin=0, nd=128, options=o)
    with Matcher(0, hbm_budget=mib << 20) as small:
        for _ in range(3):
            got = small.match(*images, dmin=0, nd=128, options=o)
            assert got.aggregate_launches >= 2 * SCANS
            for k in ("disparity", "confidence"):
                assert torch.equal(getattr(got, k).view(torch.int32), getattr(ref, k).view(torch.int32))


def test_tight_budget_hierarchy(hip_runtime, gpu):  # noqa: F811
    """The same with label ranges: ranges of few tiles, of sizes that differ
    from level to level."""
    from regard3d_mvs_amd.native import Matcher
    p = synth.make_pair(800, 600, 128, 5)
    ref = gpu.match(p.left, p.right, dmin=0, nd=128)
    for mib in (60, 75, 106):
        with Matcher(0, hbm_budget=mib << 20) as small:
            for _ in range(2):
                got = small.match(p.left, p.right, dmin=0, nd=128)
                same_bits(got.disparity, ref.disparity)
                same_bits(got.confidence, ref.confidence)


# Two levels: sweeps take the fine one from three tiles on (one and its mirror
# leave most of the device idle), with uint16 slices from six, and none wider
# than their 1024 columns.
@pytest.mark.parametrize("w,h,tile,p2,fine", [(150, 90, 512, 200, SCANS), (150, 90, 80, 200, SWEEPS),
                                              (150, 90, 80, 300, SWEEPS), (150, 70, 80, 300, SCANS),
                                              (1040, 30, 2048, 200, SCANS)])
def test_ranged_form(gpu, w, h, tile, p2, fine):  # noqa: F811
    p = synth.make_pair(w, h, 32, 11)
    g, _ = _match_both(gpu, p.left, p.right, None, None, 0, 32,
                       StereoOptions(levels=1, p2=p2, p2_adapt=0, tile_size=tile, tile_margin=4, tile_blend=4))
    assert g.aggregate_launches == (FULL if p2 <= 255 else SCANS) + fine


def test_cut_levels_by_path_scans(hip_runtime, gpu):  # noqa: F811
    """A budget that cuts the fine level into ranges of few tiles: path scans,
    in ranges of five times the cells that sweeps would take."""
    from regard3d_mvs_amd.native import Matcher
    p = synth.make_pair(1280, 960, 96, 5)
    o = StereoOptions(levels=1)
    ref = gpu.match(p.left, p.right, dmin=0, nd=96, options=o)
    assert ref.aggregate_launches == FULL + SWEEPS
    with Matcher(0, hbm_budget=600 << 20) as small:
        got = small.match(p.left, p.right, dmin=0, nd=96, options=o)
    assert got.aggregate_launches in (FULL + SCANS, 2 * FULL + SCANS)  # the coarse level may be cut in two
    same_bits(got.disparity, ref.disparity)
    same_bits(got.confidence, ref.confidence)


def test_rows_far_apart(hip_runtime, gpu):  # noqa: F811
    """Device views whose rows lie 80 MB apart: 70 of them span more than 32
    bits of offsets, which full-range scans do not hold."""
    import torch
    rng = np.random.default_rng(67)
    left = rng.integers(0, 65536, (70, 90)).astype(np.uint16)
    right = np.roll(left, -7, 1)
    o = StereoOptions(levels=0, **RAW)
    ref = gpu.match(left, right, dmin=0, nd=32, options=o)
    base = torch.empty((70, 40_000_000), dtype=torch.uint16, device="cuda")
    views = []
    for k, a in enumerate((left, right)):
        v = base[:, 1000 * k:1000 * k + 90]
        v.copy_(torch.from_numpy(a).cuda())
        views.append(v)
    got = gpu.match(*views, dmin=0, nd=32, options=o)
    assert (ref.aggregate_launches, got.aggregate_launches) == (FULL, SCANS)
    same_bits(got.disparity.cpu().numpy(), ref.disparity)
    same_bits(got.confidence.cpu().numpy(), ref.confidence)


# Scanlines about the length of the sets of loads that a full-range scan keeps
# in flight (eight), and twice that.
@pytest.mark.parametrize("short", [6, 7, 8, 9, 14, 15, 16])
@pytest.mark.parametrize("across", [False, True])
def test_full_range_short_scanlines(gpu, short, across):  # noqa: F811
    rng = np.random.default_rng(short)
    shape = (37, short) if across else (short, 37)
    left = rng.integers(0, 65536, shape).astype(np.uint16)
    right = rng.integers(0, 65536, shape).astype(np.uint16)
    g, _ = _match_both(gpu, left, right, None, None, -8, 32, StereoOptions(levels=0, **RAW))
    assert g.aggregate_launches == FULL
