"""OccupancyTable (cusync_amd/csrc/occupancy_table.h), host code only: each kernel is asked once for each size of LDS, however the
sizes take turns; an error is not remembered; more LDS than a launch may have is no workgroup, without a question."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include "occupancy_table.h"
int main() {
  cusync::rt::OccupancyTable<3, 159> table;
  int asked = 0;
  auto ask = [&](size_t bytes) { asked++; return (int)(160 * 1024 / bytes); };
  const size_t sizes[] = {64 * 1024, 100 * 1024, 147 * 1024, 64 * 1024 + 1, 159 * 1024};
  for (int turn = 0; turn < 10; turn++)
    for (int k = 0; k < 3; k++)
      for (size_t s : sizes) {
        const int want = (int)(160 * 1024 / ((s + 1023) / 1024 * 1024));
        if (table.perCU(k, s, ask) != want) { std::printf("kernel %d, %zu bytes\n", k, s); return 1; }
      }
  if (asked != 15) { std::printf("asked %d times\n", asked); return 1; }
  if (table.perCU(0, 159 * 1024 + 1, ask) != 0 || table.perCU(2, (size_t)-2048, ask) != 0 || asked != 15) { std::printf("too much LDS\n"); return 1; }
  if (table.perCU(1, 4096, [](size_t) { return -1; }) != -1 || table.perCU(1, 4096, [](size_t) { return 0; }) != 0 || table.perCU(1, 4096, ask) != 0) { std::printf("an error, none\n"); return 1; }
  if (table.perCU(1, 0, [](size_t) { return 1000; }) != 126) { std::printf("many\n"); return 1; }
  return 0;
}
"""


def test_each_size_is_asked_for_once(tmp_path):
    (tmp_path / "table.cpp").write_text(SRC)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "cusync_amd", "csrc"), str(tmp_path / "table.cpp"), "-o", str(tmp_path / "table")])
    out = subprocess.run([str(tmp_path / "table")], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
