// Choice of the number of k-slices for a GEMM of a chain, shared by the chains that make it.
#pragma once

#include <stdint.h>
#include <algorithm>

#include "../../include/cusync_amd.h"

namespace cusync {
namespace gemm {

// k-slices for a GEMM of `tiles` output tiles: double while the launch stays
// within one workgroup per CU (256 of them) and every slice keeps at least eight
// K chunks.  Small batches are bound by streaming the weights, and without
// slices a 32-row problem occupies 48 workgroups on 256 CUs; a launch of more
// than one round of workgroups pays more for adding the slices' partial sums than
// the extra loads in flight gain (M=16, N=6144, K=12288 on 32x128 tiles, 48 of them: 51 / 36 / 41 / 46 us
// with 2 / 4 / 8 / 16 slices; M=64, N=5504, K=8192 on 64x128 tiles, 43 of them: 34 / 29 / 34 / 41 us).
// Every slice takes ceil(chunks / slices) chunks of K, so a count that does not divide the chunks can leave the
// last slices without any (44 chunks in 16 slices: three each, and the sixteenth would begin past the end).
inline bool everySliceHasAChunk(uint32_t K, uint32_t bk, uint32_t slices) {
  const uint32_t chunks = (K + bk - 1) / bk;
  return slices >= 1 && slices <= chunks && (slices - 1) * ((chunks + slices - 1) / slices) < chunks;
}

// Columns of K in a slice, and whether they come in whole numbers of `unit`.
inline bool sliceInUnits(uint32_t K, uint32_t bk, uint32_t slices, uint32_t unit) {
  return ((K + bk - 1) / bk + slices - 1) / slices * bk % unit == 0;
}

// The number of columns of K a slice has to be a whole number of: 64 for the 256x384x32 tile, which refuses others.  (768 output
// columns at 1100 rows are ten of its tiles, and two slices of K = 1088 would have 17 chunks of 32 each.)
inline uint32_t sliceUnit(int tile) { return tile == CUSYNC_TILE_256x384x32 ? 64 : 1; }

inline int pickSplit(int requested, uint32_t tiles, uint32_t K, uint32_t bk, int resident, uint32_t unit = 1) {
  if (requested > 0) return requested;
  const uint32_t target = (uint32_t)std::min(resident, 256);
  int s = 1;
  while (tiles * (uint32_t)s * 2 <= target && K / ((uint32_t)s * 2) >= 8 * bk && everySliceHasAChunk(K, bk, (uint32_t)s * 2) &&
         sliceInUnits(K, bk, (uint32_t)s * 2, unit)) s *= 2;
  return s;
}

// Rounds a launch of `workgroups` takes under a limit of `cap` of them (0: no limit, one round).
inline uint32_t roundsOf(uint32_t workgroups, uint32_t cap) { return cap ? (workgroups + cap - 1) / cap : 1; }

// The same for GEMMs whose columns do not come in powers of two (the attention chain's QKV projection: 36 column tiles of
// 128, 24 of 192).  Doubling stops at half to three quarters of the CUs there, so single slices are added until four
// fifths of the CUs have work.  From eight slices on it does not pay: what they add up grows with every slice (48 rows on
// 64x192 tiles, 24 of them: 31.9 / 32.3 / 33.1 us with 8 / 9 / 10).  QKV projection, doubling -> this: 16 rows (36 tiles, 4 -> 6
// slices) 29.7 -> 26.0 us, 128 rows (48, 4 -> 5) 43.9 -> 40.5, 190 rows (72, 2 -> 3) 67.4 -> 51.9, 768 rows (72, 2 -> 3)
// 108.0 -> 93.7; level between four and seven slices once 200 CUs are busy (36 tiles, 16 rows: 26.9 / 26.0 / 26.1 us with 5 / 6 / 7).
// Nor from four slices on where the tiles have 128 rows and more and the slices share the reduction: five of them share it
// unevenly (48 tiles, the attention chain in stream order: 256 rows 102.6 us with four, 106.6 with five; 512 rows 137.5, 141.5).
// (An added slice is a whole number of 64 columns of K long whatever the tile.)
// `cap`: the caller's limit of workgroups for the launch, 0 without one.  Under a limit a slice is added only where the rounds
// it costs leave less work behind one another.  LLaMA MLP, GEMM1 of 43 tiles, 40 rows under RowSync, four slices / five: at
// most 200 workgroups, where the fifth is a second round, 50.2 / 55.8 us; 100, three rounds of fifths, 62 / 67; 160, two
// rounds either way, 61.6 / 56.6.
inline int pickSplitToFill(uint32_t tiles, uint32_t tileM, uint32_t K, uint32_t bk, int resident, uint32_t unit = 1, uint32_t cap = 0) {
  const uint32_t target = (uint32_t)std::min(resident, 256);
  uint32_t s = (uint32_t)pickSplit(0, tiles, K, bk, resident, unit);
  if (tileM >= 128 && s >= 4) return (int)s;
  for (uint32_t more = s + 1; s < 8 && tiles * s * 5 < target * 4 && more < 8 && tiles * more <= target && K / more >= 8 * bk; more++)
    if (everySliceHasAChunk(K, bk, more) && sliceInUnits(K, bk, more, 64) && roundsOf(tiles * more, cap) * s < roundsOf(tiles * s, cap) * more) s = more;
  return (int)s;
}

// Whether 256x384 tiles in three slices take over from 256x192 tiles in one: where the 256x192 tiles are too many for two
// slices on 256 CUs and leave a fifth of them or more idle in one (137 to 170 of them), half as many tiles in three slices
// keep four fifths or more busy, with two thirds of the work each and less of it loads.  `tiles`: of 256x384.  GEMMs of
// 256x192 -> 256x384, us: 12 288 to 4 608 columns (12 tiles of 384), 1300 rows 186 -> 154, 1500: 190 -> 167, 1700: 200 -> 194;
// to 6 144 columns, 1100 rows 191 -> 172, 1280: 200 -> 181.  Outside that range it falls behind (6 144 columns, 1500 rows, 96
// tiles in two slices: 215 -> 220).  The launch takes its slice count from pickSplitToFill, which has to make it three: with
// K below 768 or three slices that are not whole numbers of 64 columns it gives one or two, which is another launch than the
// one measured.  Under a limit of workgroups the slices have to be ahead by rounds as well, two thirds of
// the work in each (1100 rows, 80 tiles, the pair, 256x192 in one slice / this: at most 200 workgroups 386 / 468 us, 160: 384 / 428, 128:
// 532 / 429, 64: 694 / 632; at 100, where the rounds are level, 522 / 501, and 513 / 548 where GEMM2 has the limit too).
inline bool wideInThreeSlices(uint32_t tiles, uint32_t K, int resident, uint32_t cap = 0) {
  return resident >= 256 && tiles * 3 <= 256 && tiles * 3 * 5 >= 256 * 4 && tiles * 2 * 2 > 256 && K % 64 == 0 && 2 * roundsOf(tiles * 3, cap) < 3 * roundsOf(tiles * 2, cap) &&
         pickSplitToFill(tiles, 256, K, 32, resident, 64, cap) == 3;
}

// Whether a GEMM that consumes another's tiles in the same launch gains from fetching its weights ahead of the wait, for which
// all producer tiles of a k-slice are waited for at once (DmaCfg::AHEAD).  Under a policy that can be waited for chunk by chunk
// a long slice begins on the first chunks while the last are still being made, and that is worth more: MLPs of 32x128 and
// 64x192 tiles in one launch, TileSync and StridedSync, us with -> without, by columns of K in a slice of GEMM2: 688 43.7 -> 44.6,
// 1536 47.4 -> 48.4 and 79.8 -> 81.2, 2304 100.7 -> 101.7; 2752 113.0 -> 112.2, 3072 68.9 -> 68.5 and 121.0 -> 120.5, 4608 94.1 ->
// 93.4, 6144 116.6 -> 115.1 and 214.4 -> 210.5, 12288 214.5 -> 210.4.
inline bool fetchAheadPays(bool waitsPerChunk, uint32_t kPerSlice) { return !waitsPerChunk || kPerSlice <= 2560; }

// Whether the k-slices of a tile add it up together (each waits for its siblings, then sums and stores a share of
// the tile) instead of leaving all of it to the slice that arrives last.  The waiting slices hold their CUs, so
// every slice of the launch must have a workgroup of its own from the start (one round, all of them dealt a
// static first tile).  Where something keeps a sibling off the device for long, the tile is given up and added up by
// the last arriver after all (DynStage::gatherSlices).  Under AvoidWaitKernel that would be the rule, since the
// consumer's launch can reach the device before its producer's and take the slots the siblings need: there the
// last-arriver form is kept, whose workgroups retire at once.  Tiles of 128 rows and more with a 32-row piece for
// every slice only.
inline bool slicesCanShareReduction(int splitK, bool requested, bool directToLdsTile, bool everyTileStatic, uint32_t launched,
                                    uint32_t tiles, uint32_t tileM, bool avoidWaitKernel) {
  return splitK > 1 && requested && directToLdsTile && everyTileStatic && launched == tiles && tileM >= 128 &&
         tileM / 32 >= (uint32_t)splitK && !avoidWaitKernel;
}
// The same in equal shares, which none of the kernels needs.
inline bool slicesShareReduction(int splitK, bool requested, bool directToLdsTile, bool everyTileStatic, uint32_t launched,
                                 uint32_t tiles, uint32_t tileM, bool avoidWaitKernel) {
  return slicesCanShareReduction(splitK, requested, directToLdsTile, everyTileStatic, launched, tiles, tileM, avoidWaitKernel) &&
         (tileM / 32) % (uint32_t)splitK == 0;
}

}  // namespace gemm
}  // namespace cusync
