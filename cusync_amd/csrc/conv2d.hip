// Sync-aware NHWC forward convolution as an implicit GEMM
//   [N*P*Q, R*S*C] x [R*S*C, K]  ->  y[N,P,Q,K],   k = (r*S + s)*C + c,
// cross-correlation, fp16 in, fp32 accumulate, fp16 out, optional ReLU.
// Stands in for cutlass::conv::device::CuSyncImplicitGemmConvolution
// (src/include/cutlass/cusync-cutlass/include/cutlass/conv/device/cusyncimplicit_gemm_convolution.h:226-298)
// and its kernel (conv/kernel/implicit_cusyncgemm_convolution.h:287-477,
// conv/threadblock/implicit_cusyncgemm_pipelined.h:313-492).
//
// The kernel is the direct-to-LDS GEMM kernel with two changes: the A operand is
// gathered (a K chunk of a row is one contiguous run of channels of one input
// pixel, or zeros outside the image), and B — the KRSC filter — is already
// k-contiguous, so its stage is laid out like A's and read without transpose.
// A consumer convolution waits for every producer row block that the filter's
// halo reaches, not only for the block of its own rows.
#include <hip/hip_runtime.h>

#include <string.h>
#include <algorithm>
#include <mutex>
#include <vector>

#include "../../include/cusync_amd.h"
#include "rt_internal.h"
#include "gemm_kernel_dma.h"
#include "conv3x3_kernel.h"
#include "conv3x3_solo_kernel.h"
#include "conv3x3_rows_kernel.h"
#include "split_choice.h"
#include "occupancy_table.h"

namespace {

using namespace cusync::gemm;

struct ConvTile {
  uint32_t bm, bn, bk;
  uint32_t threads;
  size_t lds;
  void (*kernel)(GemmParams);
  void (*chainKernel)(ConvChainParams);     // several layers in one launch; halo tiles only
  void (*splitKernel)(GemmParams);          // the same tile with its steps cut into runs (split_k > 1); halo tiles only
  uint32_t (*haloLds)(uint32_t W, uint32_t C);      // a launch's LDS for images of width W with C channels; halo tiles only
};

#define CUSYNC_CONV_TILE(BM, BN, BK, WM, WN, ST, OCC) \
  { BM, BN, BK, kThreads, (size_t)DmaCfg<BM, BN, BK, WM, WN, ST, OCC, true>::LDS_BYTES, \
    gemmDmaKernel<DmaCfg<BM, BN, BK, WM, WN, ST, OCC, true>, kAConv>, nullptr, nullptr, nullptr }
#define CUSYNC_SOLO_TILE(CFG) \
  { CFG::BM, 2 * CFG::BN, CFG::BK, CFG::THREADS, 0, convHaloSoloKernel<CFG, false>, nullptr, convHaloSoloKernel<CFG, true>, CFG::ldsBytes }
#define CUSYNC_HALO_TILE(CFG) \
  { CFG::BM, CFG::BN, CFG::BK, CFG::THREADS, 0, convHalo3x3Kernel<CFG>, convHalo3x3ChainKernel<CFG>, convHalo3x3Kernel<CFG, true>, CFG::ldsBytes }

using HaloA = Halo3x3Cfg<256, 64, 4, 1, 4, 2>;     // 64 output channels per tile: four waves of 64 x 64 stacked
using HaloB = Halo3x3Cfg<128, 128, 2, 2, 3, 2, 2>;    // 128 output channels per tile
using HaloC = Halo3x3Cfg<64, 128, 2, 2, 3, 2, 2>;     // 64 pixels: what fits beside the halo of 512-channel pixels (7 x 7 images)
using HaloCPair = Halo3x3Cfg<64, 128, 2, 2, 3, 2>;    // the same tile where two of them fit a CU (convTileFor)

using Solo128 = HaloSoloCfg<128, 2, 1>;     // 64 columns of the 128x128 and of the 64x128 tile (soloTileFor)
using Solo64 = HaloSoloCfg<64, 2, 1>;
constexpr int kHaloCPair = CUSYNC_CONV_TILE_COUNT, kSolo128 = kHaloCPair + 1, kSolo64 = kHaloCPair + 2, kConvKernels = kHaloCPair + 3;
ConvTile g_convTiles[kConvKernels] = {
  CUSYNC_CONV_TILE(128, 64, 32, 2, 2, 4, 3),    // CUSYNC_CONV_TILE_128x64x32
  CUSYNC_CONV_TILE(128, 128, 32, 2, 2, 4, 2),   // CUSYNC_CONV_TILE_128x128x32
  CUSYNC_CONV_TILE(256, 64, 32, 4, 1, 3, 2),    // CUSYNC_CONV_TILE_256x64x32
  // the halo tiles: 3x3 / pad 1 / stride 1 only; LDS size depends on the image width and channels
  CUSYNC_HALO_TILE(HaloA),      // CUSYNC_CONV_TILE_HALO_256x64x64
  CUSYNC_HALO_TILE(HaloB),      // CUSYNC_CONV_TILE_HALO_128x128x64
  CUSYNC_HALO_TILE(HaloC),      // CUSYNC_CONV_TILE_HALO_64x128x64
  CUSYNC_HALO_TILE(HaloCPair),
  CUSYNC_SOLO_TILE(Solo128),
  CUSYNC_SOLO_TILE(Solo64),
};

bool isHalo(int tile) { return tile >= 0 && tile < CUSYNC_CONV_TILE_COUNT && g_convTiles[tile].haloLds; }
uint32_t haloLds(int tile, uint32_t W, uint32_t C) { return g_convTiles[tile].haloLds(W, C); }
constexpr uint32_t kMaxLds = 160 * 1024 - 1024;      // what one workgroup may ask for (the kernel has 8 bytes of static LDS)

// The halo kernel needs 3x3, pad 1, stride 1, a power-of-two channel count of at least 64, and its tile plus
// halo in LDS.  (Two lines of pixels first: of images wider than that the bytes of the halo can wrap around 32 bits.)
bool haloEligible(int tile, uint32_t W, uint32_t C, uint32_t R, uint32_t S, uint32_t pad, uint32_t stride) {
  return R == 3 && S == 3 && pad == 1 && stride == 1 && C >= 64 && (C & (C - 1)) == 0 && (uint64_t)W * C * 4 <= kMaxLds && haloLds(tile, W, C) <= kMaxLds;
}

std::mutex g_convMutex;

ConvTile* convTile(int tile) {
  if (tile < 0 || tile >= CUSYNC_CONV_TILE_COUNT) return nullptr;
  return &g_convTiles[tile];
}

// The kernels that images of width W with C channels run with.  The 64x128 tile has one group of four wavefronts where
// two tiles fit a CU's LDS (64 channels, and 128 up to a width of 28): the other tile's wavefronts then fill the gaps
// that the second group is there for, and a CU holds one tile of two groups only (with runs its kernel has 217 registers
// per lane, and the launches of a tile share one count).  One convolution, one group / two groups, in us: 32x28x28x64 to
// 64 channels 11.6 / 18.9, 32x56x56x64 35.6 / 49.8, 32x28x28x128 to 128 17.2 / 26.0; with fewer tiles than CUs level at
// 64 channels and 4 to 5 % behind at 128.  (The 128x128 tile at 64 channels, where two fit as well, is level: two groups
// from 4 % ahead to 4 % behind.)
ConvTile* convTileFor(int tile, uint32_t W, uint32_t C) {
  if (tile == CUSYNC_CONV_TILE_HALO_64x128x64 && 2 * (HaloCPair::ldsBytes(W, C) + 1024) <= 160 * 1024) return &g_convTiles[kHaloCPair];
  return convTile(tile);
}

int g_convNumCUs = 0;
cusync::rt::OccupancyTable<kConvKernels, kMaxLds / 1024> g_convOccupancy;
bool g_convLdsAllowed[kConvKernels] = {};

// Whether all kernels of a tile may ask for the LDS they will (set once).
bool allowConvLds(const ConvTile* ti) {
  bool& allowed = g_convLdsAllowed[ti - g_convTiles];
  if (allowed) return true;
  const int most = ti->haloLds ? (int)kMaxLds : (int)ti->lds;
  const void* kernels[3] = {reinterpret_cast<const void*>(ti->kernel), reinterpret_cast<const void*>(ti->chainKernel), reinterpret_cast<const void*>(ti->splitKernel)};
  for (const void* k : kernels)
    if (k && CUSYNC_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, most))) return false;
  return allowed = true;
}

// Workgroups of a tile's launches, with `lds` bytes, that the device holds at once; 0 after an error.
int residentConv(ConvTile* ti, size_t lds) {
  std::lock_guard<std::mutex> lock(g_convMutex);
  if (g_convNumCUs == 0) {
    int dev = 0;
    hipDeviceProp_t prop;
    if (CUSYNC_HIP(hipGetDevice(&dev)) || CUSYNC_HIP(hipGetDeviceProperties(&prop, dev))) return 0;
    g_convNumCUs = prop.multiProcessorCount;
  }
  if (!allowConvLds(ti)) return 0;
  const int perCU = g_convOccupancy.perCU((int)(ti - g_convTiles), lds, [ti](size_t bytes) {
    // the chain kernel is the same code in a loop, the split kernel the same with its steps in runs: the least of the three
    int least = 0, n = 0;
    if (CUSYNC_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&least, ti->kernel, (int)ti->threads, bytes))) return -1;
    if (ti->chainKernel) {
      if (CUSYNC_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, ti->chainKernel, (int)ti->threads, bytes))) return -1;
      least = std::min(least, n);
    }
    if (ti->splitKernel) {
      if (CUSYNC_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, ti->splitKernel, (int)ti->threads, bytes))) return -1;
      least = std::min(least, n);
    }
    return least;
  });
  return std::max(0, perCU) * g_convNumCUs;
}

// The kernel of conv3x3_solo_kernel.h, where a tile's split_k workgroups can be its two halves of columns times one, two or four
// runs and every one of the launch's `parts` has a workgroup from the start; null elsewhere (three runs, five, a cap, several
// rounds: the tile's own kernel with its steps in runs).  Where both can run, this one is ahead at every size measured: pairs
// under RowSync, us, runs -> this, 128x128 tile in two 1x14x14x256 45 -> 33, 32x14x14x256 47 -> 36, in four 8x14x14x256 39.2 -> 34.0;
// 64x128 tile in two 32x7x7x512 49.6 -> 42.2, in four 16x7x7x512 40.3 -> 37.1, in eight 2x7x7x512 34.4 -> 30.4; one convolution by
// itself, 128x128 tile, 4x28x28x64 in two, four and eight 13.9 -> 9.4, 14.4 -> 11.4, 17.2 -> 12.2, and nowhere behind at 64 to 512 channels.
// Not under AvoidWaitKernel (`opts`): its caller has seen to it that all stages fit on the device at once, by the tile and what
// cusync_conv2d_max_resident says of it, and here a workgroup has a CU to itself.
ConvTile* soloTileFor(int tile, int split, uint32_t parts, uint32_t W, uint32_t C, int opts) {
  if (opts & CUSYNC_OPT_AVOID_WAIT_KERNEL) return nullptr;
  if ((split != 2 && split != 4 && split != 8) || (tile != CUSYNC_CONV_TILE_HALO_128x128x64 && tile != CUSYNC_CONV_TILE_HALO_64x128x64)) return nullptr;
  ConvTile* ti = &g_convTiles[tile == CUSYNC_CONV_TILE_HALO_128x128x64 ? kSolo128 : kSolo64];
  const uint32_t lds = ti->haloLds(W, C);
  return lds <= kMaxLds && parts <= (uint32_t)residentConv(ti, lds) ? ti : nullptr;
}

using RowsKernel = void (*)(GemmParams);
RowsKernel rowsKernel(int epilogue) { return epilogue == CUSYNC_EPILOGUE_RELU ? convRowsKernel<CUSYNC_EPILOGUE_RELU> : convRowsKernel<CUSYNC_EPILOGUE_NONE>; }

// The device's CUs, once convRowsKernel has its LDS allowance; 0 after an error.
int rowsCUs() {
  static const int cus = [] {
    int dev = 0;
    hipDeviceProp_t prop;
    if (CUSYNC_HIP(hipGetDevice(&dev)) || CUSYNC_HIP(hipGetDeviceProperties(&prop, dev))) return 0;
    for (int epilogue : {CUSYNC_EPILOGUE_NONE, CUSYNC_EPILOGUE_RELU})
      if (CUSYNC_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(rowsKernel(epilogue)), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds))) return 0;
    return prop.multiProcessorCount;
  }();
  return cus;
}

// Rows of the product per workgroup of convRowsKernel (conv3x3_rows_kernel.h) for a layer of 64 channels, a workgroup per CU: whole
// sixteens, no fewer than four wavefronts have work for; 0 where its input tile and the filter do not fit the LDS.
// `overlapped`: the layers' launches go beside each other.  Where a workgroup for each CU comes out, which happens at whole multiples of
// 4096 rows, a run is sixteen rows longer: a consumer finds no CU free otherwise and is held back by the host until all of its producer
// has started, layer by layer (16x16 images under RowSync, us, 256 workgroups / this: 20 480 rows, two layers 29.9 / 24.3, four 57.1 / 42.4;
// 32 768 rows, where the sixteen are a turn more of each wavefront, 29.8 / 25.7 and 57.6 / 44.8; 98 304 rows 32.2 / 32.5 and 61.1 / 57.5).
uint32_t rowsPerWorkgroup(uint32_t N, uint32_t H, uint32_t W, bool overlapped) {
  const uint32_t M = N * H * W, cus = (uint32_t)rowsCUs();
  if (!cus) return 0;
  uint32_t rows = std::max<uint32_t>(ConvRowsCfg::WAVES * ConvRowsCfg::T, ((M + cus - 1) / cus + ConvRowsCfg::T - 1) / ConvRowsCfg::T * ConvRowsCfg::T);
  if (overlapped && (M + rows - 1) / rows >= cus && ConvRowsCfg::ldsBytes(rows + ConvRowsCfg::T, W) <= kMaxLds) rows += ConvRowsCfg::T;      // (the kernel itself is the same for every sync)
  return ConvRowsCfg::ldsBytes(rows, W) <= kMaxLds ? rows : 0;
}

// A launch's LDS for images of width W with C channels.
size_t launchLds(const ConvTile* ti, uint32_t W, uint32_t C) { return ti->haloLds ? ti->haloLds(W, C) : ti->lds; }

uint32_t outExtent(uint32_t in, uint32_t filter, uint32_t pad, uint32_t stride) { return (in + 2 * pad - filter) / stride + 1; }

size_t partialBytes(const cusync_conv2d_args* a, const ConvTile* ti) {
  const cusync_dim3 g = cusync_conv2d_grid_split(a->tile, a->N, a->H, a->W, a->K, a->R, a->S, a->pad, a->stride, a->split_k);
  return (size_t)g.z * g.y * g.x * ti->bm * ti->bn * sizeof(float);
}

// Where the workgroups of a tile hand over to one another: partial sums, and counters that are 0 between launches.
struct ConvScratch {
  void* partials;
  size_t bytes;
  void* counters;
};

bool isSolo(const ConvTile* ti) { return ti == &g_convTiles[kSolo128] || ti == &g_convTiles[kSolo64]; }

// What a caller's workspace holds: [split_k][row tiles][column tiles][BM * BN] fp32 partial sums, then two counters per output
// tile, as the GEMM's.
ConvScratch workspaceOf(const cusync_conv2d_args* a, const ConvTile* ti) {
  if (a->split_k <= 1) return {};
  const size_t bytes = partialBytes(a, ti);
  return {a->workspace, bytes, (char*)a->workspace + bytes};
}

// Kernel parameters of one convolution launched with `launched` workgroups.
GemmParams convParams(const cusync_conv2d_args* a, const ConvTile* ti, uint32_t launched, const ConvScratch& scratch) {
  const cusync_stage_desc& s = a->stage;
  GemmParams p = {};
  p.stage.d = s;
  p.cvN = a->N; p.cvH = a->H; p.cvW = a->W; p.cvC = a->C;
  p.cvP = outExtent(a->H, a->R, a->pad, a->stride);
  p.cvQ = outExtent(a->W, a->S, a->pad, a->stride);
  p.cvR = a->R; p.cvS = a->S; p.cvPad = a->pad; p.cvStride = a->stride;
  p.M = a->N * p.cvP * p.cvQ; p.N = a->K; p.K = a->R * a->S * a->C;
  p.A = (const half_t*)a->x; p.lda = a->C;
  p.B = (const half_t*)a->w; p.ldb = p.K;
  p.D = (half_t*)a->y; p.ldd = a->K;
  p.epilogue = a->epilogue;
  p.a_mode = CUSYNC_A_PLAIN;
  p.launched = launched;
  p.splitK = (uint32_t)std::max(1, a->split_k);
  const uint32_t chunks = (p.K + ti->bk - 1) / ti->bk;
  p.kPerSlice = (chunks + p.splitK - 1) / p.splitK * ti->bk;
  p.mPad = s.grid.y * ti->bm;
  p.waitRound = 1;
  p.coopReduce = 0;
  p.partials = (float*)scratch.partials;
  p.partialBytes = (uint32_t)scratch.bytes;
  p.arrivals = (uint32_t*)scratch.counters;
  cusync::rt::timeline(&p.timeline, &p.timelineCap);
  // Producer tiles are whole 128-byte lines of the activation tensor when a pixel's channels are.
  p.stage.lineAligned = !cusync::rt::forceAcquire() && s.in.kind != CUSYNC_POLICY_NOSYNC && (uintptr_t)a->x % 128 == 0 &&
                        (a->C * 2) % 128 == 0 &&
                        (s.in.kind == CUSYNC_POLICY_ROWSYNC || (s.in.tileN * 2) % 128 == 0);
  p.stage.releaseAll = cusync::rt::forceRelease();
  p.stage.prepare(launched);
  return p;
}

// One launch; the arguments are checked.  `resident`: residentConv of the kernel and these bytes of LDS.
cusync_error launchConv(const cusync_conv2d_args* a, ConvTile* ti, int resident, const ConvScratch& scratch, hipStream_t stream) {
  if (resident <= 0) { cusync::rt::setError("conv2d: kernel does not fit on a CU"); return CUSYNC_ERROR_DEVICE; }
  const uint32_t tiles = a->stage.grid.x * a->stage.grid.y * a->stage.grid.z;
  uint32_t launched = std::min<uint32_t>(tiles, (uint32_t)resident);
  if (a->max_workgroups > 0) launched = std::min<uint32_t>(launched, (uint32_t)a->max_workgroups);
  GemmParams p = convParams(a, ti, launched, scratch);
  const bool split = a->split_k > (isSolo(ti) ? 2 : 1);
  hipLaunchKernelGGL(split ? ti->splitKernel : ti->kernel, dim3(launched), dim3(ti->threads), launchLds(ti, a->W, a->C), stream, p);
  if (CUSYNC_HIP(hipGetLastError())) return CUSYNC_ERROR_DEVICE;
  cusync::rt::noteLaunch(a->stage, launched >= (uint32_t)resident);
  return CUSYNC_SUCCESS;
}

}  // namespace

extern "C" {

int cusync_conv2d_tile_shape(int tile, uint32_t* tileM, uint32_t* tileN, uint32_t* tileK) {
  ConvTile* ti = convTile(tile);
  if (!ti) return 1;
  if (tileM) *tileM = ti->bm;
  if (tileN) *tileN = ti->bn;
  if (tileK) *tileK = ti->bk;
  return 0;
}

cusync_dim3 cusync_conv2d_grid_split(int tile, uint32_t N, uint32_t H, uint32_t W, uint32_t K, uint32_t R, uint32_t S,
                                     uint32_t pad, uint32_t stride, int split_k) {
  cusync_dim3 g = {0, 0, 0};
  ConvTile* ti = convTile(tile);
  if (!ti || stride == 0 || H + 2 * pad < R || W + 2 * pad < S) return g;
  const uint32_t M = N * outExtent(H, R, pad, stride) * outExtent(W, S, pad, stride);
  g.x = (K + ti->bn - 1) / ti->bn;
  g.y = (M + ti->bm - 1) / ti->bm;
  g.z = (uint32_t)std::max(1, split_k);
  return g;
}

cusync_dim3 cusync_conv2d_grid(int tile, uint32_t N, uint32_t H, uint32_t W, uint32_t K, uint32_t R, uint32_t S,
                               uint32_t pad, uint32_t stride) {
  return cusync_conv2d_grid_split(tile, N, H, W, K, R, S, pad, stride, 1);
}

size_t cusync_conv2d_workspace_size(const cusync_conv2d_args* a) {
  ConvTile* ti = a ? convTile(a->tile) : nullptr;
  if (!ti || a->split_k <= 1) return 0;
  const cusync_dim3 g = cusync_conv2d_grid_split(a->tile, a->N, a->H, a->W, a->K, a->R, a->S, a->pad, a->stride, a->split_k);
  return partialBytes(a, ti) + 2 * (size_t)g.x * g.y * sizeof(uint32_t);
}

cusync_error cusync_conv2d_can_implement(const cusync_conv2d_args* a) {
  using cusync::rt::setError;
  if (!a) return CUSYNC_ERROR_NOT_INITIALIZED;
  ConvTile* ti = convTile(a->tile);
  if (!ti) { setError("conv2d: unknown tile id"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  if (!a->N || !a->H || !a->W || !a->C || !a->K || !a->R || !a->S || !a->stride) { setError("conv2d: empty problem"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  if (a->H + 2 * a->pad < a->R || a->W + 2 * a->pad < a->S) { setError("conv2d: filter larger than the padded image"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  if (a->pad >= a->R || a->pad >= a->S) { setError("conv2d: padding must be smaller than the filter"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  if (a->C % ti->bk) { setError("conv2d: channels must be a multiple of the K chunk"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  if (isHalo(a->tile) && !haloEligible(a->tile, a->W, a->C, a->R, a->S, a->pad, a->stride)) {
    setError("conv2d: the halo tile needs a 3x3 filter, pad 1, stride 1, a power-of-two channel count >= 64 and its rows plus 2W + 2 pixels in LDS");
    return CUSYNC_ERROR_NOT_INITIALIZED;
  }
  if (a->K % 8) { setError("conv2d: output channels must be a multiple of 8"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  const uint64_t outRows = (uint64_t)((a->H + 2 * a->pad - a->R) / a->stride + 1) * ((a->W + 2 * a->pad - a->S) / a->stride + 1) * a->N;
  if ((uint64_t)a->N * a->H * a->W * a->C * 2 >= 0x80000000ull || (uint64_t)a->K * a->R * a->S * a->C * 2 >= 0x80000000ull ||
      outRows * a->K * 2 >= 0x80000000ull) {
    setError("conv2d: operand larger than 2 GiB is not addressable by one buffer descriptor");
    return CUSYNC_ERROR_NOT_INITIALIZED;
  }
  if (((uintptr_t)a->x | (uintptr_t)a->w | (uintptr_t)a->y) % 16) { setError("conv2d: misaligned operand"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  if (a->epilogue < 0 || a->epilogue > CUSYNC_EPILOGUE_RELU) { setError("conv2d: unknown epilogue"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  if (a->split_k > 1) {
    if (!ti->splitKernel) { setError("conv2d: split_k > 1 needs a halo tile"); return CUSYNC_ERROR_NOT_INITIALIZED; }
    if ((uint32_t)a->split_k > a->R * a->S * (a->C / ti->bk)) { setError("conv2d: more runs than steps (9 * C / 64)"); return CUSYNC_ERROR_NOT_INITIALIZED; }
    if (!a->workspace || (uintptr_t)a->workspace % 16) { setError("conv2d: split_k > 1 needs a 16-byte aligned workspace of cusync_conv2d_workspace_size bytes"); return CUSYNC_ERROR_NOT_INITIALIZED; }
    if (partialBytes(a, ti) >= 0x80000000ull) { setError("conv2d: partial sums larger than 2 GiB"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  }
  const cusync_dim3 g = cusync_conv2d_grid_split(a->tile, a->N, a->H, a->W, a->K, a->R, a->S, a->pad, a->stride, a->split_k);
  const cusync_stage_desc& s = a->stage;
  if (s.grid.x != g.x || s.grid.y != g.y || s.grid.z != g.z) { setError("conv2d: stage grid does not match cusync_conv2d_grid_split"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  if (!s.tileOrder || !s.tileCounter || !s.startCounter || !s.spinTimeouts || !s.xcdTickets) { setError("conv2d: stage not allocated"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  if (s.out.kind != CUSYNC_POLICY_NOSYNC && !s.tileStatusWrite) { setError("conv2d: producer stage without semaphores"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  if (s.in.kind != CUSYNC_POLICY_NOSYNC) {
    if (!s.tileStatusRead) { setError("conv2d: consumer stage not paired with a producer"); return CUSYNC_ERROR_NOT_INITIALIZED; }
    if (s.in.tileM == 0 || s.in.tileN == 0) { setError("conv2d: input policy with zero tile extent"); return CUSYNC_ERROR_NOT_INITIALIZED; }
    if (s.in.kind != CUSYNC_POLICY_ROWSYNC && a->C / std::max(s.in.tileN, 1u) > 32) { setError("conv2d: more than 32 producer channel tiles"); return CUSYNC_ERROR_NOT_INITIALIZED; }
    if (s.in.kind == CUSYNC_POLICY_CONV2DTILESYNC && (s.in.R != a->R || s.in.S != a->S)) { setError("conv2d: Conv2DTileSync built for another filter size"); return CUSYNC_ERROR_NOT_INITIALIZED; }
  }
  if ((s.opts & CUSYNC_OPT_NO_ATOMIC_ADD) && s.out.kind != CUSYNC_POLICY_NOSYNC &&
      cusync::dyn::waitValue(s.out) != cusync::dyn::postValue(s.out)) {
    setError("conv2d: NoAtomicAdd needs a policy whose wait value equals its post value");
    return CUSYNC_ERROR_NOT_INITIALIZED;
  }
  return CUSYNC_SUCCESS;
}

int cusync_conv2d_max_resident(int tile) {
  ConvTile* ti = convTileFor(tile, 56, 64);
  if (!ti) return 0;
  return residentConv(ti, launchLds(ti, 56, 64));     // the halo tiles: for 56 x 56 x 64 images
}

cusync_error cusync_conv2d_run(const cusync_conv2d_args* a, void* stream) {
  cusync_error e = cusync_conv2d_can_implement(a);
  if (e != CUSYNC_SUCCESS) return e;
  const uint32_t tiles = a->stage.grid.x * a->stage.grid.y * a->stage.grid.z;
  const bool capped = a->max_workgroups > 0 && (uint32_t)a->max_workgroups < tiles;
  ConvTile* ti = capped ? nullptr : soloTileFor(a->tile, a->split_k, tiles, a->W, a->C, a->stage.opts);
  if (!ti) ti = convTileFor(a->tile, a->W, a->C);
  return launchConv(a, ti, residentConv(ti, launchLds(ti, a->W, a->C)), workspaceOf(a, ti), (hipStream_t)stream);
}

}  // extern "C"

/* ---- chain of same-shape 3x3 convolutions ------------------------------------------ */

struct cusync_conv_chain {
  cusync_conv_chain_config cfg;
  std::vector<const void*> w;
  std::vector<cusync_stage_desc> st;
  std::vector<hipStream_t> stream;
  std::vector<hipEvent_t> done;      // behind the run's last launch on each stream (see rt::waitEnd)
  void* ws = nullptr;                // the layers' scratch: all counters, then all partial sums
  size_t counterBytes = 0, partialBytes = 0;      // of a layer
  ConvTile* kernel = nullptr;        // what a layer runs where each has a launch of its own and it is not by rows
  int resident = 0;
  int splitK = 1;
  uint32_t rows = 0;                 // rows of the product per workgroup of convRowsKernel, 0: the tile's own kernel
  uint32_t timeoutsSeen = 0;         // sum of the stages' give-up counters when the last run returned
  bool broken = false;               // a run failed behind a launch (see rt::abandonRun)
};

namespace {

// After the runs of a call have been synchronised with: an error if a wait of any layer gave up meanwhile.
cusync_error chainTimeouts(cusync_conv_chain* c) {
  std::vector<const cusync_stage_desc*> stages;
  for (const auto& d : c->st) stages.push_back(&d);
  return cusync::rt::checkSpinTimeouts(stages.data(), (int)stages.size(), &c->timeoutsSeen, "conv chain");
}

cusync_policy_desc noSyncDesc() {
  cusync_policy_desc p;
  memset(&p, 0, sizeof p);
  p.kind = CUSYNC_POLICY_NOSYNC;
  p.tileM = p.tileN = 1; p.R = p.S = 1;
  return p;
}

ConvScratch scratchOf(const cusync_conv_chain* c, uint32_t layer) {
  char* ws = (char*)c->ws;
  if (!ws) return {};
  return {c->partialBytes ? ws + c->cfg.layers * c->counterBytes + layer * c->partialBytes : nullptr, c->partialBytes, ws + layer * c->counterBytes};
}

// One layer by rows (conv3x3_rows_kernel.h).  The arguments are checked.
cusync_error runRows(const cusync_conv2d_args* a, uint32_t rows, const ConvScratch& scratch, hipStream_t stream) {
  const uint32_t launched = (a->N * a->H * a->W + rows - 1) / rows;
  GemmParams p = convParams(a, convTile(a->tile), launched, scratch);
  p.kPerSlice = rows;
  hipLaunchKernelGGL(rowsKernel(a->epilogue), dim3(launched), dim3(ConvRowsCfg::THREADS), ConvRowsCfg::ldsBytes(rows, a->W), stream, p);
  if (CUSYNC_HIP(hipGetLastError())) return CUSYNC_ERROR_DEVICE;
  cusync::rt::noteLaunch(a->stage, launched >= (uint32_t)rowsCUs());
  return CUSYNC_SUCCESS;
}

void freeChain(cusync_conv_chain* c) {
  for (auto s : c->stream) (void)hipStreamSynchronize(s);
  for (auto& d : c->st) cusync_stage_free(&d);
  if (c->ws) (void)hipFree(c->ws);
  for (auto e : c->done) (void)hipEventDestroy(e);
  for (auto s : c->stream) (void)hipStreamDestroy(s);
  delete c;
}

}  // namespace

extern "C" {

cusync_conv_chain* cusync_conv_chain_create(const cusync_conv_chain_config* cfg, const void* const* weights) {
  using cusync::rt::setError;
  if (!cfg || !weights) { setError("conv chain: null argument"); return nullptr; }
  if (cfg->layers < 1 || cfg->layers > 16) { setError("conv chain: 1 to 16 layers"); return nullptr; }
  cusync_conv_chain* c = new cusync_conv_chain();
  c->cfg = *cfg;
  // The built-in choice, 128 channels and more: two workgroups to a tile, its halves of columns (soloTileFor), where all of the
  // launch are resident; 64 rows a tile before 128, which leaves fewer CUs idle and makes each workgroup's serial way shorter
  // (pairs under RowSync, us, 128 -> 64 rows: 1x14x14x256 32.8 -> 26.2, 20x14x14x256 34.5 -> 30.7, 8x28x28x128 27.8 -> 24.5).  Tiles of
  // 512 channels are cut into runs as well while every one still has a workgroup and 18 units (2x7x7x512 34.2 -> 30.5 in four
  // runs a half, 16x7x7x512 40.8 -> 37.1 in two); at 256 channels a cut costs in the exchange what it saves (8x14x14x256 27.2 -> 28.4).
  // Under AvoidWaitKernel neither this nor the rows below: both take a CU for each of more workgroups than the tile's own
  // kernel has (a pair of 8x28x28x128 is 392 of them and fits as 196), and a consumer that comes first would hold its producer's.
  // (Whatever the sync, so that results do not depend on it.)
  const int givenOpts = cfg->opts >= 0 ? cfg->opts : 0;
  const bool ownKernels = !(givenOpts & CUSYNC_OPT_AVOID_WAIT_KERNEL) && !(cfg->fused && cfg->sync != CUSYNC_SYNC_STREAM);
  c->splitK = 0;
  if (c->cfg.tile < 0 && cfg->split_k == 0 && ownKernels && cfg->C % 128 == 0) {
    for (int tile : {CUSYNC_CONV_TILE_HALO_64x128x64, CUSYNC_CONV_TILE_HALO_128x128x64}) {
      const cusync_dim3 g = cusync_conv2d_grid_split(tile, cfg->N, cfg->H, cfg->W, cfg->C, 3, 3, 1, 1, 2);
      if (g.x * g.y == 0 || !haloEligible(tile, cfg->W, cfg->C, 3, 3, 1, 1) || !soloTileFor(tile, 2, g.x * g.y * g.z, cfg->W, cfg->C, givenOpts)) continue;
      c->cfg.tile = tile; c->splitK = 2;
      const uint32_t units = 9 * (cfg->C / 64);
      while (units > 36 && c->splitK < 8 && units / c->splitK >= 18 && soloTileFor(tile, c->splitK * 2, g.x * g.y * c->splitK * 2, cfg->W, cfg->C, givenOpts)) c->splitK *= 2;
      break;
    }
  }
  if (c->cfg.tile < 0)
    c->cfg.tile = cfg->C % 128 == 0 && haloEligible(CUSYNC_CONV_TILE_HALO_128x128x64, cfg->W, cfg->C, 3, 3, 1, 1) ? CUSYNC_CONV_TILE_HALO_128x128x64
                  : haloEligible(CUSYNC_CONV_TILE_HALO_256x64x64, cfg->W, cfg->C, 3, 3, 1, 1) ? CUSYNC_CONV_TILE_HALO_256x64x64
                  : cfg->C % 128 == 0 && haloEligible(CUSYNC_CONV_TILE_HALO_64x128x64, cfg->W, cfg->C, 3, 3, 1, 1) ? CUSYNC_CONV_TILE_HALO_64x128x64
                  : cfg->C % 128 == 0 ? CUSYNC_CONV_TILE_128x128x32 : CUSYNC_CONV_TILE_256x64x32;
  // 64 channels, the built-in choice: tiles of 256 rows for the policies, the rows themselves dealt evenly to the CUs.
  if (cfg->tile < 0 && cfg->split_k <= 1 && cfg->C == ConvRowsCfg::CHANNELS && c->cfg.tile == CUSYNC_CONV_TILE_HALO_256x64x64 && ownKernels) {
    c->rows = rowsPerWorkgroup(cfg->N, cfg->H, cfg->W, cfg->sync != CUSYNC_SYNC_STREAM && cfg->layers > 1);
    c->splitK = 1;
  }
  uint32_t tm = 0, tn = 0;
  if (cusync_conv2d_tile_shape(c->cfg.tile, &tm, &tn, nullptr)) { setError("conv chain: unknown tile id"); delete c; return nullptr; }
  if (c->cfg.fused && cfg->sync != CUSYNC_SYNC_STREAM &&
      (!isHalo(c->cfg.tile) || cfg->layers > (uint32_t)kMaxFusedLayers || !haloEligible(c->cfg.tile, cfg->W, cfg->C, 3, 3, 1, 1))) {
    setError("conv chain: one launch for all layers needs a halo tile that fits and at most 8 layers");
    delete c;
    return nullptr;
  }
  cusync_dim3 g = cusync_conv2d_grid(c->cfg.tile, cfg->N, cfg->H, cfg->W, cfg->C, 3, 3, 1, 1);
  if (g.x == 0 || g.y == 0) { setError("conv chain: empty shape"); delete c; return nullptr; }
  // What is left for runs: a tile that the caller gives, AvoidWaitKernel, and layers whose halo fits beside the tile kernel's ring of filter
  // stages but not beside the 64 KB of the kernel above (512 channels, images 15 and 16 wide).  Where their tiles leave most of the device
  // idle the 9 * C / 64 steps of a tile are cut into runs, a workgroup each, whose partial sums are put together as the GEMM's
  // k-slices are: as many runs as stay resident together, of at least nine steps each (pairs in us without runs -> with, all under
  // AvoidWaitKernel or with the tile given: 32x14x14x256 63 -> 54 in two; 32x7x7x512 82 -> 59 in two; 8x14x14x256 65 -> 50 in four;
  // 1x7x7x512 82 -> 43 in eight; with shorter runs the exchange costs more than the idle CUs: 1x56x56x64 35 -> 50
  // in nine runs of one step), and at 128 rows a tile two or four of them.
  if (cfg->split_k > 0) c->splitK = cfg->split_k;
  else if (c->splitK == 0 && isHalo(c->cfg.tile) && !(c->cfg.fused && cfg->sync != CUSYNC_SYNC_STREAM)) {
    ConvTile* ti = convTileFor(c->cfg.tile, cfg->W, cfg->C);
    const int resident = residentConv(ti, ti->haloLds(cfg->W, cfg->C));
    const uint32_t tiles = g.x * g.y, steps = 9 * (cfg->C / 64);
    uint32_t s = resident > 0 && tiles * 2 <= (uint32_t)g_convNumCUs ? std::min<uint32_t>((uint32_t)resident / tiles, steps / 9) : 1u;
    if (tm >= 128) s = s >= 4 ? 4 : s == 3 ? 2 : s;
    while (s > 1 && (steps + s - 1) / s * (s - 1) >= steps) s--;      // no run without steps
    c->splitK = (int)std::max(1u, s);
  }
  c->splitK = std::max(1, c->splitK);
  if (c->splitK > 1 && (!isHalo(c->cfg.tile) || (c->cfg.fused && cfg->sync != CUSYNC_SYNC_STREAM))) {
    setError("conv chain: cutting a tile's steps into runs needs a halo tile and one launch per layer");
    delete c;
    return nullptr;
  }
  if (c->splitK > 1 && (uint32_t)c->splitK > 9 * (cfg->C / 64)) {
    setError("conv chain: more runs than a tile has steps (9 * C / 64)");
    delete c;
    return nullptr;
  }
  g.z = (uint32_t)c->splitK;

  // Edge policies: what a layer posts and what the next one waits on
  // (src/ml-bench/volta_conv2d/resnet.cu:107-116; in vgg.cu the middle layers are consumer and producer at once).
  cusync_policy_desc post = noSyncDesc(), wait = noSyncDesc();
  int opts = 0;
  switch (cfg->sync) {
    case CUSYNC_SYNC_STREAM:
      break;
    case CUSYNC_SYNC_ROW:
      post.kind = CUSYNC_POLICY_ROWSYNC; post.order = CUSYNC_ORDER_TRANSPOSE_XY;
      post.tileM = tm; post.tileN = 1; post.waitValue = g.x; post.postValue = 1;
      wait = post;
      opts = CUSYNC_OPT_REORDER_TILE_LOADS;      // the filters are the chain's own inputs, written by no layer
      break;
    case CUSYNC_SYNC_TILE:
      post.kind = CUSYNC_POLICY_TILESYNC; post.order = CUSYNC_ORDER_TRANSPOSE_XY;
      post.tileM = tm; post.tileN = tn; post.waitValue = 1; post.postValue = 1;
      wait = post;
      wait.kind = CUSYNC_POLICY_CONV2DTILESYNC; wait.R = 3; wait.S = 3;
      opts = CUSYNC_OPT_NO_ATOMIC_ADD | CUSYNC_OPT_REORDER_TILE_LOADS;
      break;
    default:
      setError("conv chain: sync must be STREAM, ROW or TILE");
      delete c;
      return nullptr;
  }
  if (cfg->opts >= 0) opts |= cfg->opts;
  // (Asked for the same way as cusync_conv2d_run does; an error or a tile that does not fit shows there or in the checks of a run)
  c->kernel = soloTileFor(c->cfg.tile, c->splitK, g.x * g.y * g.z, cfg->W, cfg->C, opts);
  if (!c->kernel) c->kernel = convTileFor(c->cfg.tile, cfg->W, cfg->C);
  c->resident = residentConv(c->kernel, launchLds(c->kernel, cfg->W, cfg->C));
  // Counters, and what is added up through memory: nothing by rows and where two halves of columns share a tile, half a tile for each
  // run of a half, a tile for each run.  Only the counters have to begin as 0.  In front of the stages: the copies that these make on the
  // same stream are waited for, so the counters are 0 when a run begins on the chain's own streams.
  if (c->splitK > 1 || c->rows) {
    const size_t tiles = (size_t)g.x * g.y;
    c->counterBytes = ((c->rows ? 1 : 2) * tiles * sizeof(uint32_t) + 127) / 128 * 128;
    if (!c->rows && !(isSolo(c->kernel) && c->splitK == 2))
      c->partialBytes = tiles * c->splitK * tm * (isSolo(c->kernel) ? tn / 2 : tn) * sizeof(float);
    if (CUSYNC_HIP(hipMalloc(&c->ws, cfg->layers * (c->counterBytes + c->partialBytes))) || CUSYNC_HIP(hipMemset(c->ws, 0, cfg->layers * c->counterBytes))) {
      freeChain(c);
      return nullptr;
    }
  }
  c->st.resize(cfg->layers);
  for (uint32_t i = 0; i < cfg->layers; i++) memset(&c->st[i], 0, sizeof c->st[i]);
  for (uint32_t i = 0; i < cfg->layers; i++) {
    c->w.push_back(weights[i]);
    cusync_stage_desc& d = c->st[i];
    d.grid = g; d.tileSize = {1, 1, 1}; d.iter = 1; d.opts = opts;
    d.in = i == 0 ? noSyncDesc() : wait;
    d.out = i + 1 == cfg->layers ? noSyncDesc() : post;
    if (!weights[i] || cusync_stage_create(&d, CUSYNC_ORDER_TRANSPOSE_XY) != CUSYNC_SUCCESS) { freeChain(c); return nullptr; }
  }
  if (cfg->sync != CUSYNC_SYNC_STREAM)
    for (uint32_t i = 0; i + 1 < cfg->layers; i++)
      if (cusync_set_producer_consumer_pair(&c->st[i], &c->st[i + 1]) != CUSYNC_SUCCESS) { freeChain(c); return nullptr; }
  const uint32_t streams = cfg->sync == CUSYNC_SYNC_STREAM ? 1 : cfg->layers;
  for (uint32_t i = 0; i < streams; i++) {
    hipStream_t s;
    if (CUSYNC_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking))) { freeChain(c); return nullptr; }
    c->stream.push_back(s);
    hipEvent_t e;
    if (CUSYNC_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming))) { freeChain(c); return nullptr; }
    c->done.push_back(e);
  }
  // all layers in one launch: the last one's end is the launch's
  const bool oneLaunch = c->cfg.fused && cfg->sync != CUSYNC_SYNC_STREAM;
  c->st[0].flags |= CUSYNC_STAGE_STAMPS_START;
  for (uint32_t i = 0; i < cfg->layers; i++)
    if (!oneLaunch || i + 1 == cfg->layers) c->st[i].flags |= CUSYNC_STAGE_STAMPS_END;
  return c;
}

void cusync_conv_chain_destroy(cusync_conv_chain* c) {
  if (c) freeChain(c);
}

cusync_error cusync_conv_chain_run(cusync_conv_chain* c, const void* x, void* const* ys, int runs,
                                   double* times_us, double* layer_us) {
  if (!c || !x || !ys) return CUSYNC_ERROR_NOT_INITIALIZED;
  if (c->broken) return cusync::rt::refuseBroken("conv chain");
  const uint32_t n = c->cfg.layers;
  const bool overlapped = c->cfg.sync != CUSYNC_SYNC_STREAM;
  auto layerArgs = [&](uint32_t i) {
    cusync_conv2d_args a;
    memset(&a, 0, sizeof a);
    a.stage = c->st[i];
    a.N = c->cfg.N; a.H = c->cfg.H; a.W = c->cfg.W; a.C = c->cfg.C; a.K = c->cfg.C;
    a.R = a.S = 3; a.pad = 1; a.stride = 1;
    a.x = i == 0 ? x : ys[i - 1];
    a.w = c->w[i];
    a.y = ys[i];
    a.epilogue = (c->cfg.relu && i + 1 < n) ? CUSYNC_EPILOGUE_RELU : CUSYNC_EPILOGUE_NONE;
    a.tile = c->cfg.tile;
    a.split_k = c->splitK;
    a.workspace = c->splitK > 1 ? c->ws : nullptr;      // (for the checks)
    return a;
  };
  for (uint32_t i = 0; runs > 0 && i < n; i++) {      // before anything is launched
    const cusync_conv2d_args a = layerArgs(i);
    const cusync_error e = cusync_conv2d_can_implement(&a);
    if (e != CUSYNC_SUCCESS) return e;
  }
  auto failed = [&](cusync_error why) { return cusync::rt::abandonRun(c->stream.data(), (int)c->stream.size(), &c->broken, why); };
  if (overlapped && c->cfg.fused) {
    // all layers in one launch on the first stream
    ConvTile* ti = convTileFor(c->cfg.tile, c->cfg.W, c->cfg.C);
    const size_t lds = ti->haloLds(c->cfg.W, c->cfg.C);
    const int resident = residentConv(ti, lds);
    if (resident <= 0) { cusync::rt::setError("conv chain: kernel does not fit on a CU"); return CUSYNC_ERROR_DEVICE; }
    const cusync_dim3& g = c->st[0].grid;
    const uint32_t launched = std::min<uint32_t>(g.x * g.y * g.z, (uint32_t)resident);
    for (int r = 0; r < runs; r++) {
      ConvChainParams cp = {};
      cp.layers = n;
      for (uint32_t i = 0; i < n; i++) {
        const cusync_conv2d_args a = layerArgs(i);
        cp.layer[i] = convParams(&a, ti, launched, {});
      }
      hipLaunchKernelGGL(ti->chainKernel, dim3(launched), dim3(ti->threads), lds, c->stream[0], cp);
      if (CUSYNC_HIP(hipGetLastError()) || CUSYNC_HIP(hipEventRecord(c->done[0], c->stream[0]))) return failed(CUSYNC_ERROR_DEVICE);
      const cusync_error e = cusync::rt::waitEnd(c->st[n - 1], c->stream[0], "conv chain");
      if (e != CUSYNC_SUCCESS) return failed(e);
      if (times_us) times_us[r] = cusync::rt::stampsUs(c->st[0], false, c->st[n - 1]);
      for (uint32_t i = 0; i < n; i++) c->st[i].iter += 1;
    }
    return chainTimeouts(c);
  }
  for (int r = 0; r < runs; r++) {
    for (uint32_t i = 0; i < n; i++) {
      hipStream_t s = c->stream[overlapped ? i : 0];
      const cusync_conv2d_args a = layerArgs(i);
      cusync_error e;
      // overlapped: layer i's stream is held back until layer i - 1 is on the device: by the reference's wait kernel
      // where that layer's launch left workgroup slots free (32x56x56x64: 251 workgroups on 256 CUs), so that the wait
      // kernel's wave takes nothing from the producer; from this thread where the launch took them all.
      if (overlapped && i > 0 && (e = cusync_hold_back(&c->st[i - 1], s)) != CUSYNC_SUCCESS) return failed(e);
      e = c->rows ? runRows(&a, c->rows, scratchOf(c, i), s) : launchConv(&a, c->kernel, c->resident, scratchOf(c, i), s);
      if (e != CUSYNC_SUCCESS) return i ? failed(e) : e;
    }
    for (uint32_t i = 0; i < (overlapped ? n : 1); i++) if (CUSYNC_HIP(hipEventRecord(c->done[i], c->stream[i]))) return failed(CUSYNC_ERROR_DEVICE);
    for (uint32_t i = n; i-- > (overlapped ? 0 : n - 1);) {
      const cusync_error e = cusync::rt::waitEnd(c->st[i], c->stream[overlapped ? i : 0], "conv chain");
      if (e != CUSYNC_SUCCESS) return failed(e);
    }
    if (times_us) times_us[r] = cusync::rt::stampsUs(c->st[0], false, c->st[n - 1]);
    if (!overlapped && layer_us)
      for (uint32_t i = 0; i < n; i++) layer_us[(size_t)r * n + i] = cusync::rt::stampsUs(c->st[i ? i - 1 : 0], i > 0, c->st[i]);
    for (uint32_t i = 0; i < n; i++) c->st[i].iter += 1;
  }
  return chainTimeouts(c);
}

const cusync_stage_desc* cusync_conv_chain_stage(const cusync_conv_chain* c, uint32_t which) {
  if (!c || which >= c->cfg.layers) return nullptr;
  return &c->st[which];
}

int cusync_conv_chain_tile(const cusync_conv_chain* c) { return c ? c->cfg.tile : -1; }
int cusync_conv_chain_split(const cusync_conv_chain* c) { return c ? c->splitK : -1; }

}  // extern "C"
