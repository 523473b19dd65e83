"""Serving admits by the bytes of the volumes that its pairs will hold."""
import time

import pytest

from regard3d_mvs_amd import StereoOptions, synth

pytestmark = pytest.mark.gpu


# A budget between one pair's estimate and two: 192 bytes a pixel of images,
# pyramids and maps, and 2.4 tile cells a pixel and label of 9.25 bytes each
# (byte planes) or 17.25 (uint16 slices), for 48 labels with ranges.
@pytest.mark.parametrize("levels,nd,p2,per_cell", [(1, 64, 200, 9.25), (1, 64, 300, 17.25), (0, 64, 200, 9.25),
                                                   (0, 64, 300, 3.25)])
def test_admission_counts_the_form_of_the_volumes(hip_runtime, levels, nd, p2, per_cell):
    from regard3d_mvs_amd.native import Matcher
    w, h = 320, 240
    pair = synth.make_pair(w, h, nd, 3)
    one = (192 + 2.4 * (48 if levels else nd) * per_cell) * w * h
    o = StereoOptions(levels=levels, p2=p2, p2_adapt=0)
    for room, allowed in ((1.9 * one, 1), (2.1 * one, 2)):
        most = 0
        with Matcher(0) as m:
            m.serve_start(o, hbm_budget=int(room))
            try:
                tickets = [m.submit(pair.left.shape, 0, nd, left=pair.left, right=pair.right) for _ in range(12)]
                while True:
                    st = m.server_stats()
                    most = max(most, st["active"])
                    if st["completed"] + st["failed"] == len(tickets):
                        break
                    time.sleep(0.0002)
                for t in tickets:
                    m.wait(t)
            finally:
                m.serve_stop()
        assert most <= allowed
