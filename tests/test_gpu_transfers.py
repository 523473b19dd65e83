"""Host images and maps of every size move staged or by DMA: padded rows in
pageable and page-locked memory, on both sides of 64 KiB and 1 MiB, give the
device tensors' result and leave the padding as it was."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(hip_runtime):
    from regard3d_mvs_amd.native import Matcher
    with Matcher(0) as m:
        yield m


def padded(a, pad, pinned):
    from regard3d_mvs_amd.native import host_empty
    shape = (a.shape[0], a.shape[1] + pad)
    full, keep = host_empty(shape, a.dtype) if pinned else (np.empty(shape, a.dtype), None)
    full[:] = 77
    view = full[:, pad // 2:pad // 2 + a.shape[1]]
    view[:] = a
    return full, view, keep


@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("pad", [0, 7])
@pytest.mark.parametrize("h,w,dtype", [(17, 33, np.uint8), (96, 128, np.uint16), (150, 220, np.uint8),
                                       (700, 801, np.uint16)])
def test_padded_rows(gpu, h, w, dtype, pad, pinned):
    import torch
    rng = np.random.default_rng(h)
    left = rng.integers(0, 256, (h, w)).astype(dtype)
    right = np.roll(left, -3, 1)
    valid = (rng.random((h, w)) < 0.9).astype(np.uint8) * 255
    tdt = torch.uint8 if dtype == np.uint8 else torch.uint16
    dev = [torch.from_numpy(a.astype(np.int32)).to(tdt).cuda() for a in (left, right)]
    want = gpu.match(dev[0], dev[1], left_valid=torch.from_numpy(valid).cuda(), nd=16)
    ins = [padded(a, pad, pinned) for a in (left, right, valid)]
    outs = [padded(np.zeros((h, w), np.float32), pad, pinned) for _ in range(2)]
    gpu.match(ins[0][1], ins[1][1], left_valid=ins[2][1], nd=16, out=(outs[0][1], outs[1][1]))
    for (full, view, _), ref in zip(outs, (want.disparity, want.confidence)):
        np.testing.assert_array_equal(view, ref.cpu().numpy())
        edge = np.concatenate([full[:, :pad // 2], full[:, pad // 2 + w:]], axis=1)
        assert (edge == 77).all()
