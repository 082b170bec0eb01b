"""How a launch hands its tiles out (cusync_amd/csrc/tile_deal.h), host code only.  With at least as many workgroups as tiles
every tile is exactly one workgroup's, whatever the grid, and the workgroups beyond the tiles get none; also where the lists are
begun some positions further on, as those of a later GEMM of one launch are.  With fewer, the places the workgroups begin with
and the draws cover every tile once."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <vector>
#include "tile_deal.h"
using namespace cusync::deal;
static int check(uint32_t gx, uint32_t gy, uint32_t gz, uint32_t more, uint32_t turn) {
  const cusync_dim3 grid = {gx, gy, gz};
  const uint32_t tiles = gx * gy * gz, launched = tiles + more;
  std::vector<int> taken(tiles, 0);
  uint32_t without = 0, inPlace = 0;
  for (uint32_t b = 0; b < launched; b++) {
    const uint32_t t = onlyTicket(grid, launched, b, turn);
    if (t == kNoTicket) { without++; continue; }
    if (t >= tiles || taken[t]++) { std::printf("grid %u %u %u + %u: ticket %u of workgroup %u\n", gx, gy, gz, more, t, b); return 1; }
    // a workgroup within its list's length begins with its list's position, as in a launch of several rounds
    if (b / 8 < listTiles(grid, b % 8)) { inPlace++; if (t != listTicket(grid, b % 8, b / 8, turn)) { std::printf("grid %u %u %u: workgroup %u is not in its list\n", gx, gy, gz, b); return 1; } }
  }
  if (without != more) { std::printf("grid %u %u %u + %u: %u workgroups without a tile\n", gx, gy, gz, more, without); return 1; }
  return 0;
}
// fewer workgroups than tiles: each begins with its place in its list, and what is left of a list is drawn from its dispenser
static int checkDraws(uint32_t gx, uint32_t gy, uint32_t gz, uint32_t launched) {
  const cusync_dim3 grid = {gx, gy, gz};
  const uint32_t tiles = gx * gy * gz;
  std::vector<int> taken(tiles, 0);
  uint32_t sum = 0;
  auto take = [&](uint32_t t) { return t < tiles && !taken[t]++; };
  for (uint32_t b = 0; b < launched; b++)
    if (b / 8 < listTiles(grid, b % 8)) { sum++; if (!take(listTicket(grid, b % 8, b / 8))) { std::printf("grid %u %u %u / %u: workgroup %u\n", gx, gy, gz, launched, b); return 1; } }
  for (uint32_t x = 0; x < 8; x++)
    for (uint32_t l = listStatic(grid, x, launched); l < listTiles(grid, x); l++) { sum++; if (!take(listTicket(grid, x, l))) { std::printf("grid %u %u %u / %u: list %u, position %u\n", gx, gy, gz, launched, x, l); return 1; } }
  if (sum != tiles) { std::printf("grid %u %u %u / %u: %u tiles\n", gx, gy, gz, launched, sum); return 1; }
  return 0;
}
int main() {
  for (uint32_t gx = 1; gx <= 40; gx++)
    for (uint32_t gy = 1; gy <= 14; gy++)
      for (uint32_t gz = 1; gz <= 5; gz++)
        for (uint32_t more : {0u, 1u, 7u, 8u, 30u})
          for (uint32_t turn : {0u, 1u, 3u})
            if (check(gx, gy, gz, more, turn)) return 1;
  for (uint32_t gx = 1; gx <= 40; gx++)
    for (uint32_t gy = 1; gy <= 14; gy++)
      for (uint32_t gz = 1; gz <= 5; gz++)
        for (uint32_t launched : {1u, 3u, 8u, 9u, 31u, 100u, 256u})
          if (launched < gx * gy * gz && checkDraws(gx, gy, gz, launched)) return 1;
  // launches of the chains: 14 x 14 x 256 at batch 32, LLaMA's GEMM1, the QKV projection, attention, one column of 392 tiles
  const uint32_t chains[][3] = {{2, 49, 2}, {29, 4, 2}, {29, 8, 1}, {36, 1, 4}, {43, 1, 4}, {12, 1, 6}, {12, 4, 2}, {1, 392, 1}, {64, 4, 1}};
  for (auto& c : chains) for (uint32_t turn = 0; turn < 8; turn++) if (check(c[0], c[1], c[2], 0, turn)) return 1;
  // the lists turn for one row of tiles with a CU for each, the weights' rows a multiple of 1 KiB apart
  const struct { bool oneRow; uint32_t tiles, launched, pitches; bool turns; } launches[] = {
    {true, 240, 240, 12288 | 24576, true}, {true, 256, 256, 12288 | 24576, true}, {true, 192, 192, 49152 | 24576, true},
    {true, 384, 384, 98304 | 24576, false}, {true, 240, 100, 12288 | 24576, false}, {false, 128, 128, 12288 | 24576, false},
    {true, 215, 215, 11008 | 16384, false}, {true, 240, 240, 12544 | 24832, false}};
  for (auto& l : launches)
    if (listsTurn(l.oneRow, l.tiles, l.launched, 256, l.pitches) != l.turns) { std::printf("turn: %u tiles, %u workgroups, pitches %u\n", l.tiles, l.launched, l.pitches); return 1; }
  std::printf("ok\n");
  return 0;
}
"""


def test_every_tile_is_one_workgroups(tmp_path):
    src = tmp_path / "tile_deal_test.cpp"
    src.write_text(SRC)
    exe = tmp_path / "tile_deal_test"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "cusync_amd", "csrc"), str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)], text=True).strip() == "ok"
