// Instantiates part of the GEMM tile table (see gemm_tiles.h).
#include "gemm_tiles.h"
#include "gemm_kernel_dma.h"

namespace cusync {
namespace gemm {

// As many workgroups to a CU as the tile's other kernels leave room for, so that two launches of several GEMMs fit the device
// together where they did: one of 32x128, whose two times 80 KB are a few bytes too many (seven stages, 120 KB of loads in
// flight: 32 rows of the LLaMA MLP of inner width 5504 70.3 -> 69.4 us against four stages, of the GPT-3 MLP 72.0 -> 71.4), two
// of 64x128 (one of six stages: 64 rows of GPT-3 83.9 -> 83.4 us, which is not worth the slot), one of 64x192.
using Chain32x128 = DmaCfgAhead<32, 128, 64, 1, 4, 7, 1>;
using Chain64x128 = DmaCfgAhead<64, 128, 64, 1, 4, 3, 2>;
using Chain64x192 = DmaCfgAhead<64, 192, 64, 2, 2, 4, 1>;

void fillDmaTilesFew(TileInfo* t) {
  t[CUSYNC_TILE_D32x128x64] = CUSYNC_TILE_DMA_FEW(Chain32x128, 32, 128, 64, 1, 4, 4, 2);     // 60 KB of loads in flight per workgroup
  t[CUSYNC_TILE_D64x128x64] = CUSYNC_TILE_DMA_FEW(Chain64x128, 64, 128, 64, 1, 4, 3, 2);
  t[CUSYNC_TILE_D64x192x64] = CUSYNC_TILE_DMA_FEW(Chain64x192, 64, 192, 64, 2, 2, 4, 1);     // 96 KB of loads in flight per CU
}

}  // namespace gemm
}  // namespace cusync
