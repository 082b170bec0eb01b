// The last GEMM of a chain with its weights held in registers ahead of the wait (gemm_resident_kernel.h): when, its grid, its launch.
#pragma once

#include "../../include/cusync_amd.h"

namespace cusync {
namespace gemm {

// K up to 1536 is what the registers hold.  Up to 112 rows: each 16 rows more cost it 1.7 us (2 with 128 columns) and the tiles none
// (12 heads, hidden 12288, under RowSync, tiles / this: 112 rows behind 2000 93.7 / 92.4, behind 4000 99.3 / 97.9; 128 rows behind 2000
// 94.6 / 95.5, behind 8000 107.7 / 108.7, without a cache 84.0 / 82.4).  Columns for half the CUs at least and one round at most: hidden
// 8192, 16 rows behind 1000 51.7 -> 47.0, 16384 68.5 -> 59.9; with 3 heads, whose K is a quarter, 39.4 -> 38.9.
inline bool weightsFitRegisters(uint32_t M, uint32_t N, uint32_t K) {
  const uint32_t tiles = (N + 63) / 64;
  return M <= 112 && K <= 1536 && tiles >= 128 && tiles <= 256;
}
// Columns of a workgroup: 64, which reads its weights in half the time, where each has a CU of its own beside the `others`
// workgroups of the stage in front of it (32 rows behind 100 under RowSync, 48 of them, 128 columns / 64: 57.2 / 56.0 us, in stream
// order 64.8 / 61.1; 64 rows without a cache 65.8 / 61.1); else 128, so that none begins when the others are done.
inline uint32_t residentColumns(uint32_t N, uint32_t others) { return (N + 63) / 64 + others <= 256 ? 64 : 128; }
inline cusync_dim3 residentGrid(uint32_t N, uint32_t columns) { return cusync_dim3{(N + columns - 1) / columns, 1, 1}; }
// `a` as for cusync_gemm_run but for the stage's grid, which is residentGrid(a->N, columns); checked by the caller.  No k-slices,
// no epilogue, a stage that posts nothing and waits, if at all, by RowSync or TileSync.
cusync_error residentRun(const cusync_gemm_args* a, uint32_t columns, void* stream);

}  // namespace gemm
}  // namespace cusync
