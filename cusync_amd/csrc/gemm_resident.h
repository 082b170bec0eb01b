// The last GEMM of a chain with its weights held in registers ahead of the wait (gemm_resident_kernel.h): when, its grid, its launch.
#pragma once

#include "../../include/cusync_amd.h"

namespace cusync {
namespace gemm {

// K up to 1536 is what the registers hold; columns for half the CUs at least and one round at most.  Each 16 rows cost it 1.7 us (2
// with 128 columns) and the tiles none until their next row tile, and the weights it has ahead of the wait are worth the more the
// longer K is; so the rows it takes over go by K, and by whether the tiles it takes the place of are the 64x192 ones, which fill the
// CUs from 65 rows on (other widths: tiles of 128 columns, which do not).  One rule for every sync, since results must not depend
// on it.  The layer, us, tiles / this, each pass on other operands than the one before, in stream order | RowSync | TileSync:
//   hidden 12288, 12 heads, 32 rows 58.7 / 57.7 | 54.3 / 53.2 | 55.3 / 51.1; 64 rows 69.8 / 65.9 | 64.9 / 60.7 | 65.9 / 60.2; 112 rows
//   85.7 / 84.9 | 83.1 / 79.7 | 86.2 / 82.1; behind 4000: 32 rows 67.0 / 66.2 | 64.2 / 60.0 | 62.0 / 57.8; 112 rows 103.3 / 103.0 | 98.3 /
//   97.8 | 98.7 / 96.5.  (On the same operands again and again, which the last-level cache then holds, the tiles are up to 6 % ahead from
//   80 rows on in stream order and 3 % under RowSync, level or behind under TileSync.)
//   hidden 9216, 5 heads, 64 rows 56.1 / 52.8 | 49.0 / 45.6 | 51.5 / 46.9; 80 rows 58.1 / 59.2 | 55.4 / 53.9 | 58.8 / 55.9
//   hidden 8192, 12 heads, 112 rows 81.3 / 74.8 | 76.7 / 68.9 | 77.4 / 71.4
//   hidden 16384, 3 heads, 16 rows 43.0 / 44.0 | 38.2 / 37.7 | 41.1 / 37.8; 32 rows 43.8 / 46.1 | 39.7 / 39.5 | 41.7 / 40.2; 48 rows 64.6 / 61.7 |
//   57.0 / 55.4 | 60.3 / 57.3
//   hidden 8192, 1 head, 16 rows 36.7 / 37.4 | 31.6 / 31.3 | 33.9 / 31.6; 32 rows 37.1 / 38.8 | 31.6 / 32.1 | 34.5 / 33.2
// The lines lie where it falls more than 3 % behind in stream order (1 to 12 heads, hidden 8192 to 16384, no cache and 2000 cached rows).
// `cus`: the device's.
inline bool weightsFitRegisters(uint32_t M, uint32_t N, uint32_t K, uint32_t cus) {
  const uint32_t tiles = (N + 63) / 64;
  if (M > 112 || K > 1536 || 2 * tiles < cus || tiles > cus) return false;
  if (N % 192 == 0) return M <= (K >= 1024 ? 112u : K >= 512 ? 64u : K >= 384 ? 16u : 0u);
  if (K >= 640) return true;
  if (M > 32) return K >= 256 || N <= 12288;
  if (M > 16) return K >= 384 && N <= 12288;       // the tiles of 32 rows do these in the time of 16
  return K >= 384 || (K >= 256 && N <= 12288) || N <= 8192;
}
// Columns of a workgroup: 64, which reads its weights in half the time, where each has a CU of its own beside the `others`
// workgroups of the stage in front of it (32 rows behind 100 under RowSync, 48 of them, 128 columns / 64: 57.2 / 56.0 us, in stream
// order 64.8 / 61.1; 64 rows without a cache 65.8 / 61.1); else 128, so that none begins when the others are done.
inline uint32_t residentColumns(uint32_t N, uint32_t others, uint32_t cus) { return (N + 63) / 64 + others <= cus ? 64 : 128; }
inline cusync_dim3 residentGrid(uint32_t N, uint32_t columns) { return cusync_dim3{(N + columns - 1) / columns, 1, 1}; }
// Gives the kernel its LDS; false after an error.  Called when a handle that will launch it is made.
bool residentReady(uint32_t columns);
// `a` as for cusync_gemm_run but for the stage's grid, which is residentGrid(a->N, columns); checked by the caller.  No k-slices,
// no epilogue, a stage that posts nothing and waits, if at all, by RowSync or TileSync.
cusync_error residentRun(const cusync_gemm_args* a, uint32_t columns, void* stream);

}  // namespace gemm
}  // namespace cusync
