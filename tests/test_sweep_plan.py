"""The row sweeps' LDS and scratch rows hold every chunk a row can have (host
arithmetic of csrc/sweep_plan.hpp; no GPU needed)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "sweep_plan.hpp"
using namespace r3dg;
int main() {
  const int lds = 160 << 10;
  for (int np : {1, 3})
    for (int w : {1, 2, 63, 113, 596, 608, 1023, 1024, 1025})
      for (int per : {1, 2, 8, 31, 32, 33, 125, 215, 216, 217, 250}) {  // chunks of every pixel
        const auto chunks = static_cast<std::uint32_t>(w * per);
        const SweepPlan p = size_sweep(np, w, chunks, chunks, 256, lds);
        std::printf("%d %d %u %d %d %d %d %d\n", np, w, chunks, p.ok, p.cap, p.swords, p.lds_bytes, p.held);
      }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++20", "-Wall", "-Werror", "-I", os.path.join(ROOT, "regard3d_mvs_amd", "csrc"),
                    str(d / "plan.cpp"), "-o", str(d / "plan")], check=True)
    out = subprocess.run([str(d / "plan")], check=True, capture_output=True, text=True).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


def test_rows_hold_every_chunk(plans):
    for np_, w, chunks, ok, cap, swords, lds_bytes, held in plans:
        assert not (ok and w > 1024)
        if not ok:
            continue
        # The last word of a row: the sentinel after the last pixel's labels.
        last = 8 * chunks + w
        assert cap > last if swords == 0 else swords > last, (np_, w, chunks)
        assert lds_bytes <= 160 << 10
        # Chunks past the held ones start past the LDS row.
        assert 8 * 1024 * held >= cap
        # What a window that is not used reads: the first ten words and none past the row's pad.
        assert cap + 8 >= 10
    # The shortest rows are taken (they all fit), and rows of more than 2^17 chunks.
    assert all(ok for _, w, chunks, ok, *_ in plans if w <= 113)
    assert any(ok and chunks > 1 << 17 for _, _, chunks, ok, *_ in plans)


FORMS = r"""
#include <cstdio>
#include "sweep_plan.hpp"
int main() {
  unsigned long long tiles, cells, cap, scan_cap;
  int bytes;
  while (std::scanf("%llu %llu %llu %llu %d", &tiles, &cells, &cap, &scan_cap, &bytes) == 5)
    std::printf("%d\n", r3dg::sweeps_fit(tiles, cells, cap, scan_cap, bytes != 0, 256) ? 1 : 0);
}
"""


def test_sweeps_fit(tmp_path):
    """Sweeps where a range has blocks enough; levels that path scans would cut
    into fewer ranges only with many."""
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    (tmp_path / "fit.cpp").write_text(FORMS)
    subprocess.run([cxx, "-std=c++20", "-Wall", "-Werror", "-I", os.path.join(ROOT, "regard3d_mvs_amd", "csrc"),
                    str(tmp_path / "fit.cpp"), "-o", str(tmp_path / "fit")], check=True)
    cases = [(2, 10, 100, 500, 1, 0), (3, 10, 100, 500, 1, 1), (5, 10, 100, 500, 0, 0), (6, 10, 100, 500, 0, 1),
             (0, 0, 100, 500, 1, 0), (96, 150, 100, 500, 1, 0), (342, 150, 100, 500, 1, 1), (341, 150, 100, 500, 1, 0),
             (700, 1050, 100, 500, 1, 0), (48, 99, 100, 500, 0, 1), (10, 10, 0, 0, 1, 0),
             (96, 150, 100, 100, 1, 1), (22, 150, 100, 100, 1, 1), (21, 150, 100, 100, 1, 0)]
    text = "".join("%d %d %d %d %d\n" % c[:5] for c in cases)
    out = subprocess.run([str(tmp_path / "fit")], input=text, check=True, capture_output=True, text=True).stdout
    assert [int(v) for v in out.split()] == [c[5] for c in cases]
