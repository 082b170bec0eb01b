// Which tile a workgroup of a persistent launch begins with: host and device code, so that it can be checked on the CPU.
//
// Each of the eight XCDs has its own L2, so which workgroup gets which tile decides how much of the operands is
// re-fetched from memory.  The tiles are therefore dealt in eight lists, one per XCD.  With at least eight column tiles
// list x holds the column tiles [x*gx/8, (x+1)*gx/8) of every row, in row-major order: its workgroups share the same few
// B column panels (and, row by row, the same A panels) in their L2.  With fewer column tiles (a convolution with 64
// output channels has one) it holds the row tiles [x*gy/8, (x+1)*gy/8) instead, so that the rows of A it reads (for a
// convolution each input pixel is read by up to R*S neighbouring rows) stay in its L2.  A ticket is the tile's position
// in the row-major schedule; it still goes through the stage's ticket -> tile table.
//
// Workgroups are dispatched to the XCDs round-robin: workgroup b works on list b % 8 and begins with position b / 8 of it.
#pragma once

#include "policy_eval.h"

namespace cusync {
namespace deal {

constexpr uint32_t kNoTicket = 0xffffffffu;

CUSYNC_HD bool byRows(const cusync_dim3& grid) { return grid.x < 8; }
CUSYNC_HD uint32_t listTiles(const cusync_dim3& grid, uint32_t x) {
  const uint32_t span = byRows(grid) ? grid.y : grid.x;
  return ((x + 1) * span / 8 - x * span / 8) * (byRows(grid) ? grid.x : grid.y) * grid.z;
}
CUSYNC_HD uint32_t listWorkgroups(uint32_t x, uint32_t launched) { return launched > x ? (launched - x + 7) / 8 : 0; }
// Positions of list x that are handed out statically to the first tiles of the workgroups.
CUSYNC_HD uint32_t listStatic(const cusync_dim3& grid, uint32_t x, uint32_t launched) {
  const uint32_t wgs = listWorkgroups(x, launched), tiles = listTiles(grid, x);
  return wgs < tiles ? wgs : tiles;
}
// Ticket of position l of list x.  `turn`: the list is begun that many positions further on (see listsTurn).
CUSYNC_HD uint32_t listTicket(const cusync_dim3& grid, uint32_t x, uint32_t l, uint32_t turn = 0) {
  if (turn) l = (l + turn) % listTiles(grid, x);
  const uint32_t span = byRows(grid) ? grid.y : grid.x;
  const uint32_t lo = x * span / 8, width = (x + 1) * span / 8 - lo;
  if (!byRows(grid)) return lo + l % width + (l / width) * grid.x;
  const uint32_t perSlice = width * grid.x;          // this list's tiles in one k-slice
  return (l / perSlice) * grid.x * grid.y + lo * grid.x + l % perSlice;
}

// Whether the later GEMMs of a launch of several begin their lists a position further on each.  A workgroup has the same
// position in each one's list, so without the turn the tiles it gets have much the same columns.  Where the rows of the
// weights are a multiple of 1 KiB apart, all rows of a column tile lie in one class of memory channels, one class in four is
// a quarter slower, and the workgroups that finish such a tile last would begin another one.  GPT-3 MLP in one launch (48 and
// 96 column tiles, lists of 6 and 12), a pass without -> with the turn, us: TileSync 1 row 70.5 -> 68.9, 16 rows 71.9 -> 70.1, 64
// rows 80.2 -> 79.8, inner width 24576, 1 row 217.3 -> 215.0; RowSync 1 row 70.9 -> 70.4, 16 rows 72.3 -> 71.5.
// Not where there are more tiles than CUs or workgroups, which costs under TileSync what is not explained (inner width 49152,
// 384 tiles: 1 row 385.6 -> 407.5, 32 rows 410.9 -> 433.6; RowSync level).  Not where several row tiles read the same weights (512 to 1024 rows: level), nor at
// other row pitches (LLaMA, 11008 bytes, StridedSync, 1 row 43.9 and 44.2, 16 rows 44.7 and 45.1: level).
// `pitches`: the row pitches of all the GEMMs' weights in bytes, or'ed.
inline bool listsTurn(bool oneRowOfTiles, uint32_t mostTiles, uint32_t launched, uint32_t numCUs, uint32_t pitches) {
  return oneRowOfTiles && mostTiles <= launched && mostTiles <= numCUs && pitches % 1024 == 0;
}

// A launch of at least as many workgroups as tiles needs no dispenser: every tile is some workgroup's first one.  Where
// the lists do not come out even (98 tiles of a convolution: lists of 12 to 14 for 12 or 13 workgroups each) the
// workgroups beyond their own list's length take, in order, the positions that other lists have left over.  Drawn from
// the dispensers instead, those workgroups began 2.5 us after the others, every workgroup paid two round trips to learn
// that nothing is left, and the k-slices of a tile could not share their reduction (slicesCanShareReduction).
CUSYNC_HD uint32_t leftOver(const cusync_dim3& grid, uint32_t launched, uint32_t b, uint32_t turn = 0) {
  const uint32_t mine = b & 7u;
  uint32_t s = b / 8 - listTiles(grid, mine);        // how many workgroups without a place of their own come before this one
  for (uint32_t x = 0; x < mine; x++) {
    const uint32_t tiles = listTiles(grid, x), wgs = listWorkgroups(x, launched);
    if (wgs > tiles) s += wgs - tiles;
  }
  for (uint32_t x = 0; x < 8; x++) {
    const uint32_t tiles = listTiles(grid, x), wgs = listWorkgroups(x, launched);
    const uint32_t left = tiles > wgs ? tiles - wgs : 0;
    if (s < left) return listTicket(grid, x, wgs + s, turn);
    s -= left;
  }
  return kNoTicket;                                  // more workgroups than tiles
}
// The only ticket of workgroup b of such a launch.
CUSYNC_HD uint32_t onlyTicket(const cusync_dim3& grid, uint32_t launched, uint32_t b, uint32_t turn = 0) {
  return b / 8 < listTiles(grid, b & 7u) ? listTicket(grid, b & 7u, b / 8, turn) : leftOver(grid, launched, b, turn);
}

// The tile of workgroup b of such a launch where only the rows matter for locality (a convolution's): the tiles in the order
// row by row, all columns and parts of a row together, are cut into eight runs whose lengths differ by one at most.  Every
// list has a tile for each of its workgroups then, and the tile is two divisions away from the index.
CUSYNC_HD cusync_dim3 evenTile(const cusync_dim3& grid, uint32_t tiles, uint32_t b) {
  const uint32_t x = b & 7u, rest = tiles & 7u, at = x * (tiles >> 3) + (x < rest ? x : rest) + (b >> 3);
  const uint32_t perRow = grid.x * grid.z;
  cusync_dim3 t;
  t.y = at / perRow;
  const uint32_t in = at - t.y * perRow;
  t.z = in / grid.x;
  t.x = in - t.z * grid.x;
  return t;
}

}  // namespace deal
}  // namespace cusync
