"""rectify_image where the row loads and shared quotients change over: sources
of one to five columns and rows, targets of odd heights, and a target focal
length whose quotients take plain divisions; bit-exact against the CPU oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from regard3d_mvs_amd import Camera, CameraModel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(hip_runtime):
    from regard3d_mvs_amd.native import Matcher
    with Matcher(0) as m:
        yield m


def check(gpu, src, cam, tgt):
    for a, b in zip(gpu.rectify(src, cam, tgt), O.rectify(src, cam, tgt)):
        np.testing.assert_array_equal(np.asarray(a).view(np.uint8), np.asarray(b).view(np.uint8))


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.float32])
@pytest.mark.parametrize("w,h", [(1, 1), (2, 7), (3, 2), (4, 4), (5, 1), (64, 3)])
def test_narrow_sources_and_odd_targets(gpu, dtype, w, h):
    rng = np.random.default_rng(w * 10 + h)
    src = (200 * rng.random((h, w))).astype(dtype)
    cam = Camera(w, h, 4.0, 4.0, (w - 1) / 2, (h - 1) / 2, CameraModel.radial_k1, (-0.02,))
    for tw, th in ((1, 1), (257, 3), (2 * w + 3, 2 * h + 4)):
        check(gpu, src, cam, Camera(tw, th, 3.7, 3.9, (tw - 1) / 2, (th - 1) / 2))


@pytest.mark.parametrize("fx", [-50.0, 1e-9, 1e41])
def test_plain_divisions(gpu, fx):
    src = np.arange(60 * 80, dtype=np.uint16).reshape(60, 80)
    cam = Camera(80, 60, 50.0, 50.0, 40.0, 30.0)
    check(gpu, src, cam, Camera(83, 61, fx, 50.0, 41.0, 30.0))
