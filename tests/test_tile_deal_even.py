"""evenTile (cusync_amd/csrc/tile_deal.h), host code only: every tile is exactly one workgroup's whatever the grid, and the tiles
of one XCD's workgroups follow one another row by row."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <vector>
#include "tile_deal.h"
int main() {
  for (uint32_t gx = 1; gx <= 12; gx++)
    for (uint32_t gy = 1; gy <= 60; gy++)
      for (uint32_t gz = 1; gz <= 8; gz++) {
        const cusync_dim3 grid = {gx, gy, gz};
        const uint32_t tiles = gx * gy * gz;
        std::vector<int> taken(tiles, 0);
        std::vector<int> last(8, -1);
        for (uint32_t b = 0; b < tiles; b++) {
          const cusync_dim3 t = cusync::deal::evenTile(grid, tiles, b);
          if (t.x >= gx || t.y >= gy || t.z >= gz || taken[t.x + gx * (t.y + gy * t.z)]++) { std::printf("grid %u %u %u: workgroup %u\n", gx, gy, gz, b); return 1; }
          const int at = (int)((t.y * gz + t.z) * gx + t.x);
          if (last[b % 8] >= 0 && at != last[b % 8] + 1) { std::printf("grid %u %u %u: workgroup %u leaves its run\n", gx, gy, gz, b); return 1; }
          last[b % 8] = at;
        }
      }
  return 0;
}
"""


def test_even_dealing_covers_every_tile_once(tmp_path):
    (tmp_path / "even.cpp").write_text(SRC)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "cusync_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                           str(tmp_path / "even.cpp"), "-o", str(tmp_path / "even")])
    out = subprocess.run([str(tmp_path / "even")], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
