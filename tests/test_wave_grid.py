"""The work split of the streaming kernels (make_wave_grid in bgk_wave.h), compiled for
the host: every strip covers its rows once and stays within what a buffer store can
address (kMaxStrip elements from the wave's first column on, or one row at any width),
and strips that run no wall's code keep T + 1 rows off the walls, on lattices from one
node to the widest that fit a device.  Runs without a GPU.
"""
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <cstdio>
#include "bgk_wave.h"
using namespace bgk::wave;
static long bad = 0, total = 0;
static void check(int nx, int ny, int T, int extra, int most, int rows) {
  if ((nx + 2.0) * (ny + 2.0) > 2.4e9) return;  // (more than 288 GB of the smallest handle)
  const int cols = kLanes - 2 * T;
  const WaveGrid g = make_wave_grid(nx, ny, cols, T, extra, 1.4, most, 256, rows);
  const int64_t room = std::max<int64_t>(1, kMaxStrip / ((int64_t)nx + 256));
  ++total;
  bool ok = g.nseg == (nx + cols - 1) / cols && g.ne <= g.nseg && g.re >= 1;
  // strips of the walls' segments: rows 1..ny in pieces of re
  ok = ok && g.re <= room && g.re <= kMaxRows && (int64_t)g.nse * g.re >= ny &&
       (int64_t)(g.nse - 1) * g.re < ny;
  int64_t edge = (int64_t)g.ne * g.nse, mid = 0;
  if (g.ne < g.nseg) {  // lowest and highest strip, and those between
    const int inner = ny - 2 * g.ra;
    ok = ok && g.ra >= T + 1 && g.ra <= room && g.rows <= room && g.rows <= kMaxRows && inner > 0 &&
         (int64_t)g.nmid * g.rows >= inner && (int64_t)(g.nmid - 1) * g.rows < inner;
    edge += 2 * (int64_t)(g.nseg - g.ne);
    mid = (int64_t)(g.nseg - g.ne) * g.nmid;
  }
  ok = ok && g.nedge == edge && g.nwg >= edge + mid && g.nwg < edge + mid + 8 &&
       (g.nwg - g.nedge) % 8 == 0;
  if (!ok && bad++ < 10)
    std::printf("nx=%d ny=%d T=%d most=%d rows=%d: nseg %d ne %d re %d nse %d ra %d rows %d\n", nx,
                ny, T, most, rows, g.nseg, g.ne, g.re, g.nse, g.ra, g.rows);
}
int main() {
  const int nxs[] = {1, 59, 60, 61, 62, 121, 185, 1003, 4096, 8192, 100000, 1000003, 16000000,
                     22369365, 22369366, 33554175, 33554176, 50000000, 67108607, 67108608,
                     134217727, 140000000, 268435456};
  const int nys[] = {1, 2, 3, 5, 6, 7, 9, 12, 40, 777, 4096};
  for (int nx : nxs)
    for (int ny : nys)
      for (int T = 1; T <= 3; ++T)
        for (int most : {16, 32, 64})
          for (int rows : {0, 1, 3, 64}) {
            check(nx, ny, T, 2 * T, most, rows);
            check(nx, ny, T, 2 * (T - 1), most, rows);
          }
  std::printf("total=%ld bad=%ld\n", total, bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_strips_cover_the_rows_within_what_a_store_addresses(tmp_path):
    src, exe = tmp_path / "t.hip", tmp_path / "t"
    src.write_text(PROGRAM)
    csrc = ROOT / "bgk_pcm_amd" / "csrc"
    subprocess.run(["hipcc", "--offload-host-only", "-O1", "-std=c++17", f"-I{csrc}", "-c",
                    str(src), "-o", str(tmp_path / "t.o")], check=True)
    subprocess.run(["hipcc", str(tmp_path / "t.o"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert "bad=0" in r.stdout
