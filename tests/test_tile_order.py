"""Which tile each workgroup of a look-back launch takes (osm::tile_order and
osm::spread_slot in orthossm_amd/csrc/osm_kernels.h), on the CPU.

Two properties.  Every tile of every lane-block is taken once.  And a block
that waits on earlier tiles of its lane-block finds their blocks already
running, whatever else occupies the GPU: they are lower-numbered blocks of the
same residue mod 8 (workgroups go to the 8 XCDs round-robin by index and in
index order within an XCD), or the tile was drawn from the lane-block's
counter when the block started.  A lower index on another XCD is not enough:
blocks of two launches could then hold the XCDs that each other's awaited
blocks need."""
import os
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SRC = r"""
#include <stdio.h>
#include <vector>
#include "osm_kernels.h"
static int check_order(int n_lb, int n_tiles, bool state_in_place) {
  const osm::TileOrder o = osm::tile_order(n_lb, n_tiles, 1, state_in_place);
  if (o.lead != (state_in_place && n_tiles > 1) || (o.lead && !o.spread)) return printf("FAIL lead n_lb=%d\n", n_lb);
  std::vector<long long> block((size_t)n_lb * n_tiles, -1);   // by index: who takes the tile
  std::vector<int> drawn(n_lb, 0);
  for (unsigned b = 0; b < o.grid; ++b) {
    osm::TileSlot s{(int)(b / n_lb), osm::slot_lane_block((int)(b % n_lb), n_lb)};
    if (o.spread) s = osm::spread_slot(o, b, n_lb, n_tiles);
    if (s.lb < 0) continue;
    if (s.lb >= n_lb || s.tile >= n_tiles) return printf("FAIL range n_lb=%d n_tiles=%d b=%u\n", n_lb, n_tiles, b);
    if (s.tile < 0) {
      if (s.lb < n_lb / 8 * 8) return printf("FAIL counter n_lb=%d lb=%d\n", n_lb, s.lb);
      ++drawn[s.lb];
      continue;
    }
    long long& at = block[(size_t)s.lb * n_tiles + s.tile];
    if (at >= 0) return printf("FAIL twice n_lb=%d n_tiles=%d lb=%d tile=%d\n", n_lb, n_tiles, s.lb, s.tile);
    at = b;
  }
  for (int lb = 0; lb < n_lb; ++lb) {
    if (drawn[lb] && drawn[lb] != n_tiles) return printf("FAIL drawn n_lb=%d n_tiles=%d lb=%d\n", n_lb, n_tiles, lb);
    for (int t = 0; t < n_tiles; ++t) {
      const long long b = block[(size_t)lb * n_tiles + t];
      if ((b >= 0) == (drawn[lb] > 0)) return printf("FAIL cover n_lb=%d n_tiles=%d lb=%d t=%d\n", n_lb, n_tiles, lb, t);
      if (t == 0 || b < 0) continue;
      const long long a = block[(size_t)lb * n_tiles + t - 1];
      if (a >= b || (a & 7) != (b & 7)) return printf("FAIL order n_lb=%d n_tiles=%d lb=%d t=%d\n", n_lb, n_tiles, lb, t);
    }
  }
  return 0;
}
static int check(int n_lb, int n_tiles) { return check_order(n_lb, n_tiles, false) || check_order(n_lb, n_tiles, true); }
int main() {
  for (int n_lb = 1; n_lb <= 70; ++n_lb)
    for (int n_tiles : {1, 2, 3, 7, 8, 9, 31, 32, 33, 40, 127, 512, 1000})
      if (check(n_lb, n_tiles)) return 1;
  for (int n_lb : {95, 96, 97, 255, 1001, 4099}) for (int n_tiles : {1, 2, 5, 64, 341}) if (check(n_lb, n_tiles)) return 1;
  if (check(1, 1 << 20) || check(9, 300001) || check(15, 100003)) return 1;
  puts("ok");
  return 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not found")
def test_every_tile_once_and_awaited_blocks_already_running():
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "t.cpp"), os.path.join(d, "t")
        with open(src, "w") as f:
            f.write(SRC)
        subprocess.run([HIPCC, "-O2", "-std=c++17", "-I", os.path.join(ROOT, "orthossm_amd", "csrc"), "-o", exe, src],
                       check=True, capture_output=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
