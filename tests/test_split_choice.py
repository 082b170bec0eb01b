"""The k-slice rule of the GEMM launcher and of the chains (cusync_amd/csrc/split_choice.h), host code only.

The kernel gives slice z the K chunks [z * per, (z + 1) * per) with per = ceil(chunks / slices): a slice count is
usable only if the last slice still begins inside K.  The closed form the library uses is checked against that
definition by brute force, and the automatic choice against the cases the design was measured on."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include "split_choice.h"
using namespace cusync::gemm;
int main() {
  // every (chunks, slices) pair of a small range: 1 if the library accepts it
  for (uint32_t chunks = 1; chunks <= 96; chunks++)
    for (uint32_t slices = 1; slices <= 40; slices++)
      std::printf("E %u %u %d\n", chunks, slices, everySliceHasAChunk(chunks * 64 - 8, 64, slices) ? 1 : 0);
  const uint32_t cases[][4] = {
    {48, 12288, 64, 256}, {96, 6144, 64, 256}, {32, 12288, 64, 256}, {64, 6144, 64, 256},     // GPT-3 shard, few rows
    {43, 8192, 64, 512}, {64, 2752, 64, 256}, {64, 2816, 64, 256},                               // LLaMA shard
    {64, 12288, 32, 256}, {128, 6144, 32, 256}, {256, 12288, 32, 256}, {512, 6144, 32, 256},    // 512 and 2048 rows on 256x192
    {1, 8256, 64, 256}, {1, 64, 64, 256}};
  for (auto& c : cases) std::printf("P %u %u %u %u %d\n", c[0], c[1], c[2], c[3], pickSplit(0, c[0], c[1], c[2], (int)c[3]));
  std::printf("R %d\n", pickSplit(7, 48, 12288, 64, 256));
  // shared reduction: (slices, requested, direct tile, all static, launched, tiles, tileM, AvoidWaitKernel)
  std::printf("S %d\n", slicesShareReduction(4, true, true, true, 256, 256, 256, false) ? 1 : 0);
  std::printf("S %d\n", slicesShareReduction(4, true, true, true, 256, 256, 256, true) ? 1 : 0);     // consumer may arrive first
  std::printf("S %d\n", slicesShareReduction(4, false, true, true, 256, 256, 256, false) ? 1 : 0);   // not asked for
  std::printf("S %d\n", slicesShareReduction(4, true, true, true, 200, 256, 256, false) ? 1 : 0);    // a second round
  std::printf("S %d\n", slicesShareReduction(4, true, true, true, 256, 256, 64, false) ? 1 : 0);     // few-row tile
  std::printf("S %d\n", slicesShareReduction(3, true, true, true, 192, 192, 256, false) ? 1 : 0);    // 8 pieces, 3 slices
  std::printf("S %d\n", slicesShareReduction(1, true, true, true, 256, 256, 256, false) ? 1 : 0);    // no slices
  std::printf("S %d\n", slicesShareReduction(2, true, false, true, 256, 256, 256, false) ? 1 : 0);   // register-staged tile
  std::printf("S %d\n", slicesShareReduction(2, true, true, false, 256, 256, 256, false) ? 1 : 0);   // tiles drawn from a dispenser
  return 0;
}
"""


def test_split_choice(tmp_path):
    src = tmp_path / "split_choice_test.cpp"
    src.write_text(SRC)
    exe = tmp_path / "split_choice_test"
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "cusync_amd", "csrc"), str(src), "-o", str(exe)])
    out = subprocess.check_output([str(exe)], text=True).split("\n")
    picks = {}
    shares = []
    for line in out:
        f = line.split()
        if not f:
            continue
        if f[0] == "E":
            chunks, slices, got = int(f[1]), int(f[2]), int(f[3])
            per = -(-chunks // slices)
            # the definition: every slice z < slices begins before the end of K (K = chunks * 64 - 8: a ragged last chunk)
            want = all(z * per * 64 < chunks * 64 - 8 for z in range(slices))
            assert got == int(want), (chunks, slices)
        elif f[0] == "P":
            picks[tuple(int(v) for v in f[1:5])] = int(f[5])
        elif f[0] == "S":
            shares.append(int(f[1]))
        elif f[0] == "R":
            assert int(f[1]) == 7                     # a requested count is passed through (and validated by the GEMM)
    # one workgroup per CU at most, and at least eight chunks per slice
    assert picks[(48, 12288, 64, 256)] == 4 and picks[(96, 6144, 64, 256)] == 2
    assert picks[(32, 12288, 64, 256)] == 8 and picks[(64, 6144, 64, 256)] == 4
    assert picks[(43, 8192, 64, 512)] == 4            # 344 workgroups would be a second round
    assert picks[(64, 2752, 64, 256)] == 4 and picks[(64, 2816, 64, 256)] == 4
    assert picks[(64, 12288, 32, 256)] == 4 and picks[(128, 6144, 32, 256)] == 2
    assert picks[(256, 12288, 32, 256)] == 1 and picks[(512, 6144, 32, 256)] == 1
    # 129 chunks: sixteen slices of nine would leave the last one empty, and the doubling stops at eight
    assert picks[(1, 8256, 64, 256)] == 8
    assert picks[(1, 64, 64, 256)] == 1
    # the slices of a tile wait for each other only where nothing can keep a sibling off the device: never for a stage
    # under AvoidWaitKernel, whose consumer may be dispatched ahead of its producer
    assert shares == [1, 0, 0, 0, 0, 0, 0, 0, 0]


FILL = r"""
#include <cstdio>
#include "split_choice.h"
using namespace cusync::gemm;
int main() {
  for (uint32_t tiles = 1; tiles <= 300; tiles++)
    for (uint32_t K : {64u, 1536u, 2752u, 6144u, 8192u, 12288u})
      for (int resident : {0, 256, 512})
        for (uint32_t tileM : {64u, 256u})
          std::printf("F %u %u %d %u %d %d\n", tiles, K, resident, tileM, pickSplit(0, tiles, K, 64, resident), pickSplitToFill(tiles, tileM, K, 64, resident));
  for (uint32_t tiles = 1; tiles <= 300; tiles++)
    for (uint32_t K = 64; K <= 16384; K += 64) {       // 32 columns of K to a chunk, as the 256x384 tile has: no slice it refuses, added or doubled
      const uint32_t unit = sliceUnit(CUSYNC_TILE_256x384x32);
      for (int got : {pickSplit(0, tiles, K, 32, 256, unit), pickSplitToFill(tiles, 256, K, 32, 256, unit), pickSplitToFill(tiles, 64, K, 32, 256, unit)})
        if ((K / 32 + got - 1) / got * 32 % 64) std::printf("B %u %u %d\n", tiles, K, got);
    }
  for (uint32_t tiles = 1; tiles <= 300; tiles++)
    for (uint32_t K = 32; K <= 16384; K += 32) {       // the launch takes its slice count from pickSplitToFill: it has to be the three the tile was chosen for
      const int got = pickSplitToFill(tiles, 256, K, 32, 256, sliceUnit(CUSYNC_TILE_256x384x32));
      if (wideInThreeSlices(tiles, K, 256) && (got != 3 || K % 64 || (K / 32 + 2) / 3 % 2)) std::printf("B %u %u %d\n", tiles, K, got);
    }
  for (uint32_t tiles = 1; tiles <= 300; tiles++)
    for (uint32_t K : {64u, 96u, 2752u, 4096u, 8192u, 12288u}) std::printf("W %u %u %d %d\n", tiles, K, wideInThreeSlices(tiles, K, 256) ? 1 : 0, wideInThreeSlices(tiles, K, 0) ? 1 : 0);
  // a limit of workgroups: never more work behind one another than without the added slices, and the tile as measured
  for (uint32_t tiles = 1; tiles <= 256; tiles++)
    for (uint32_t cap = 1; cap <= 300; cap++) {
      const uint32_t doubled = (uint32_t)pickSplit(0, tiles, 12288, 64, 256), got = (uint32_t)pickSplitToFill(tiles, 64, 12288, 64, 256, 1, cap);
      if (got != doubled && roundsOf(tiles * got, cap) * doubled >= roundsOf(tiles * doubled, cap) * got) std::printf("C %u %u %u\n", tiles, cap, got);
      if (cap >= 256 && got != (uint32_t)pickSplitToFill(tiles, 64, 12288, 64, 256)) std::printf("C %u %u %u\n", tiles, cap, got);
      if (wideInThreeSlices(tiles, 12288, 256, cap) && pickSplitToFill(tiles, 256, 12288, 32, 256, 64, cap) != 3) std::printf("C %u %u wide\n", tiles, cap);
    }
  for (uint32_t cap : {0u, 300u, 240u, 239u, 200u, 160u, 128u, 100u}) std::printf("L %u %d %d\n", cap, wideInThreeSlices(80, 12288, 256, cap) ? 1 : 0, pickSplitToFill(43, 64, 8192, 64, 256, 1, cap));
  for (uint32_t k : {64u, 688u, 1536u, 2304u, 2752u, 3072u, 12288u}) std::printf("A %u %d %d\n", k, fetchAheadPays(false, k) ? 1 : 0, fetchAheadPays(true, k) ? 1 : 0);
  for (int slices = 1; slices <= 10; slices++)
    for (uint32_t tileM : {32u, 64u, 128u, 256u})
      std::printf("S %d %u %d %d\n", slices, tileM, slicesCanShareReduction(slices, true, true, true, 240, 240, tileM, false) ? 1 : 0,
                  slicesCanShareReduction(slices, true, true, true, 240, 240, tileM, true) || slicesCanShareReduction(slices, false, true, true, 240, 240, tileM, false) ||
                  slicesCanShareReduction(slices, true, false, true, 240, 240, tileM, false) || slicesCanShareReduction(slices, true, true, false, 240, 240, tileM, false) ||
                  slicesCanShareReduction(slices, true, true, true, 200, 240, tileM, false) ? 1 : 0);
}
"""


def test_slices_that_fill_the_device(tmp_path):
    src = tmp_path / "fill_test.cpp"
    src.write_text(FILL)
    exe = tmp_path / "fill_test"
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "cusync_amd", "csrc"), str(src), "-o", str(exe)])
    lines = [f.split() for f in subprocess.check_output([str(exe)], text=True).split("\n") if f]
    fill, limits = {}, {}
    for f in lines:
        v = [int(x) for x in f[1:]]
        if f[0] == "F":
            tiles, K, resident, tileM, doubled, got = v
            fill[(tiles, K, resident, tileM)] = got
            assert doubled <= got and (got == doubled or got < 8) and (got == doubled or doubled < 4 or tileM < 128)
            if got != doubled:                                # never a second round, never without need, never a slice without work
                assert tiles * got <= min(resident, 256) and tiles * (got - 1) * 5 < min(resident, 256) * 4 and K >= 8 * 64 * got
            chunks = -(-K // 64)
            assert (got - 1) * -(-chunks // got) < chunks
        elif f[0] == "B":
            assert False, "256x384x32: slices that are not whole numbers of 64 columns, or not the three the tile was chosen for: %s" % f
        elif f[0] == "C":
            assert False, "more rounds than without the added slices: %s" % f
        elif f[0] == "A":
            assert v[1] == 1 and v[2] == int(v[0] <= 2304)        # a row is waited for as a whole; tile by tile, long slices begin early
        elif f[0] == "L":
            limits[v[0]] = (v[1], v[2])
        elif f[0] == "W":
            tiles, K, got, without = v
            per = -(-K // 32 // 3) * 32
            assert not without and (not got or (205 <= tiles * 3 <= 256 and tiles * 4 > 256 and per % 64 == 0 and 2 * per < K))
            if K == 12288:
                assert got == int(69 <= tiles <= 85)
        else:
            assert v[2] == int(1 < v[0] <= v[1] // 32 and v[1] >= 128) and not v[3]
    # the QKV projection's 36 and 24 column tiles, LLaMA's 43, and launches the doubling fills already
    want = {(36, 12288): 6, (48, 12288): 5, (72, 12288): 3, (96, 12288): 2, (24, 12288): 8, (120, 12288): 2, (43, 8192): 5, (58, 8192): 4, (64, 6144): 4}
    for (tiles, K), s in want.items():
        assert fill[(tiles, K, 256, 64)] == s, (tiles, K)
    assert fill[(48, 12288, 256, 256)] == 4 and fill[(72, 12288, 256, 256)] == 3
    # GPT-3 at five row tiles, whether in three slices of 256x384; LLaMA's 43 tiles, slices
    assert limits == {0: (1, 5), 300: (1, 5), 240: (1, 5), 239: (0, 5), 200: (0, 4), 160: (0, 5), 128: (1, 5), 100: (0, 4)}
