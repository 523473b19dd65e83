"""rectify_image of targets that see past the source, partly or all of them, so
that whole waves have no pixel inside and others few; bit-exact against the CPU
oracle."""
import numpy as np
import pytest

from regard3d_mvs_amd import Camera, CameraModel
from test_gpu_rectify_edges import check, gpu  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.float32])
@pytest.mark.parametrize("w,h", [(3, 3), (61, 47)])
@pytest.mark.parametrize("deg", [30, 70, 120])
def test_turned_targets(gpu, dtype, w, h, deg):  # noqa: F811
    rng = np.random.default_rng(deg + w)
    src = (200 * rng.random((h, w))).astype(dtype)
    if dtype is np.float32:
        src[0, 0] = src[-1, -1] = np.nan  # taps of pixels outside are not used, whatever they hold
    a = np.radians(deg)
    turn = np.array([[np.cos(a), 0, np.sin(a)], [0, 1, 0], [-np.sin(a), 0, np.cos(a)]])
    cam = Camera(w, h, 0.9 * w, 0.9 * w, (w - 1) / 2, (h - 1) / 2, CameraModel.radial_k1, (-0.02,), tuple(turn.ravel()))
    check(gpu, src, cam, Camera(517, 33, 150.0, 150.0, 200.0, 16.0))
