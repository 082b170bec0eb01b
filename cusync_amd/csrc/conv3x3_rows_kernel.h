// 3x3, pad 1, stride 1 convolution of 64 to 64 channels by rows: the filter in registers, a run of rows per CU.
//
// With 256x64 tiles, two to a CU, a layer of 32x56x56x64 is 392 tiles on 256 CUs: the CUs with two of them take twice as long as
// those with one, every tile streams the 72 KB of the filter through a ring of stages with a barrier each, and its 64 x 64 per
// wavefront read LDS as long as they multiply.  Here the rows of the product are cut into as many runs as there are CUs, of
// equal length (a multiple of 16, whatever the tiles); a wavefront holds the whole filter as fragments, 288 of its 512
// registers, and takes 16 rows at a time to all 64 columns: one LDS read for four MFMAs, and no barrier once the run's pixels
// and halo have landed.  A tile is posted by the workgroup that finishes its last rows (a count of rows per tile).
//
// Pairs, us, 256x64 tiles -> this: 1x56x56x64 under RowSync 27.6 -> 18.8, 4x 27.6 -> 21.3, 16x 31.2 -> 27.5, 32x 39.7 -> 34.3 (a
// layer's kernel alone 16 -> 11).  Longer chains: four layers 1x 47.6 -> 30.2, 16x 53.1 -> 47.3, 32x 62.0 -> 58.6; sixteen 1x 176 -> 112, 16x 180 -> 171,
// 32x 217 -> 218 (214 -> 218 on another machine; in stream order 279 -> 239): there the middle layers' workgroups, which count themselves
// started only behind their own wait, hold back the layer after them.  (Counted ahead of the wait: 8 images, four layers 44.3 -> 40.5, 32 images 58.6 ->
// 60.2.)  What bounds it at 32 images: seven times 72 MFMAs a wavefront take 7.9 us (5.1 us by themselves at the 1.95 GHz
// the device runs them at; stores 0.7, the rest issue slots, one wavefront per SIMD having all the registers), loads before them 2.6.
// 32 rows at a time (half the address arithmetic, but 13 tiles of 32 rows do not divide among four wavefronts): level there,
// 19.4 at one image.
#pragma once

#include "conv3x3_kernel.h"

namespace cusync {
namespace gemm {

// T: rows of the product (pixels) a wavefront works on at a time.
struct ConvRowsCfg {
  static constexpr int T = 16, THREADS = 256, WAVES = 4, TILE_ROWS = 256, CHANNELS = 64;
  static constexpr int KS = 32, STEPS = 9 * CHANNELS / KS, PER_TAP = CHANNELS / KS, NC = CHANNELS / T;
  static constexpr uint32_t FILTER_BYTES = CHANNELS * 9 * CHANNELS * 2;
  static constexpr uint32_t OUT_PITCH = CHANNELS * 2 + 16, OUT_BYTES = T * OUT_PITCH;
  static constexpr int AHEAD = 6;       // fragments of the input read ahead of their products
  static uint32_t haloBytes(uint32_t rows, uint32_t W) { return ((rows + 2 * W + 3) * CHANNELS * 2 + 1023) / 1024 * 1024; }
  static uint32_t ldsBytes(uint32_t rows, uint32_t W) { return FILTER_BYTES + haloBytes(rows, W); }
};

template<int EPILOGUE>
__global__ __launch_bounds__(ConvRowsCfg::THREADS, 1) void convRowsKernel(GemmParams p) {
  using C = ConvRowsCfg;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  asm volatile("" :: "s"(p.cvW), "s"(p.cvH), "s"(p.A), "s"(p.B), "s"(p.M), "s"(p.launched), "s"(p.kPerSlice), "s"(p.timeline));
  asm volatile("" :: "s"(p.stage.d.flags), "s"(p.stage.d.opts), "s"(p.stage.d.in.kind), "s"(p.stage.d.out.kind), "s"(p.stage.d.startCounter));
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t px = lane % C::T, part = lane / C::T;      // this lane's pixel, and which eight of a product's channels it holds
  const cusync::DynStage& stage = p.stage;
  const uint32_t W = p.cvW, H = p.cvH, R = p.kPerSlice;
  const bool consumer = stage.isConsumer();

  const unsigned long long tlEntry = p.timeline ? wall_clock64() : 0;
  const unsigned long long entered = stage.enter();
  // This workgroup's run of rows, [r0, r1): neighbours on one XCD, whose L2 then has their halos.
  const uint32_t list = blockIdx.x & 7u, rest = p.launched & 7u, at = list * (p.launched >> 3) + min(list, rest) + (blockIdx.x >> 3);
  const uint32_t r0 = at * R, r1 = min(p.M, r0 + R);
  const unsigned long long tl0 = p.timeline ? wall_clock64() : 0;

  const uint4v rA = rawRsrc(p.A, p.M * C::CHANNELS * 2);
  const uint4v rB = rawRsrc(p.B, C::FILTER_BYTES);
  const uint32_t ldsBase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;

  // LDS: [the run and its halo, 128 bytes a pixel, and a pixel of zeros][filter, 1152 bytes an output channel; later the rows on their
  // way out].  Chunk c of pixel n, and of each 128 bytes of channel n, at c ^ (n/2 & 7), as in conv3x3_kernel.h.
  const uint32_t haloPix = R + 2 * W + 2, haloLoads = ((haloPix + 1) * 128 + 1023) / 1024, filter = haloLoads * 1024;
  // What a wavefront loads behind the start count arrives behind it, 1 to 3 us when hundreds of workgroups count at once.  Where a
  // workgroup has little to do the consumer's launch waits for the last count, and the wavefront that counts loads nothing; where
  // it has more, the consumer waits for CUs in any case, and the count goes out behind the loads and is looked at after the first
  // tile (pairs under RowSync against stream order on the same machine: 1x56x56x64 0.97 and 1.04, 32x56x56x64 0.95 and 0.93).
  const bool early = R <= C::WAVES * C::T, counts = stage.countsStart() && wave == 0;
  const uint32_t others = early && stage.countsStart() ? 1 : 0, loaders = C::WAVES - others, loader = wave - others;       // (loader: all ones where it has nothing to load)
  uint32_t startToken = 0;
  if (early && tid == 0) stage.finishStart(stage.beginStart(), p.launched, entered);
  auto issueFilter = [&] {
    for (uint32_t q = loader; q < C::FILTER_BYTES / 1024; q += loaders) {
      const uint32_t line = q * 8 + lane / 8, n = line / 9;
      loadToLds(rB, __builtin_amdgcn_readfirstlane(ldsBase + filter + q * 1024), line * 128 + (((uint32_t)lane & 7) ^ ((n >> 1) & 7)) * 16);
    }
  };
  const bool weightsFirst = !consumer || (stage.d.opts & CUSYNC_OPT_REORDER_TILE_LOADS);
  if (weightsFirst) issueFilter();
  if (consumer) {
    const uint32_t tmq = stage.d.in.tileM, lo = r0 > W + 1 ? r0 - (W + 1) : 0, hiRow = min(r1 + W, p.M - 1);
    if (stage.d.in.kind == CUSYNC_POLICY_ROWSYNC) stage.waitWaveRows(lo, hiRow, tmq, 0, 1);
    else {
      const uint32_t tnq = stage.d.in.tileN, perTile = stage.d.in.kind == CUSYNC_POLICY_CONV2DTILESYNC ? 9 * tnq : tnq;
      for (uint32_t ct = 0; ct < C::CHANNELS / tnq; ct++) stage.waitWaveRows(lo, hiRow, tmq, ct * perTile, 0);
    }
  }
  if (!weightsFirst) issueFilter();
  for (uint32_t q = loader; q < haloLoads; q += loaders) {
    const uint32_t pl = q * 8 + lane / 8;
    const uint32_t chunk = ((uint32_t)lane & 7) ^ ((pl >> 1) & 7), flat = r0 + pl - (W + 1);
    const bool inside = r0 + pl >= W + 1 && flat < p.M && pl < haloPix;
    loadToLds(rA, __builtin_amdgcn_readfirstlane(ldsBase + q * 1024), inside ? flat * 128 + chunk * 16 : kOutOfRange);
  }
  if (!early && counts && lane == 0) startToken = stage.beginStart();
  const unsigned long long tl1 = p.timeline ? wall_clock64() : 0;

  // The filter into registers while the halo is on its way.
  const uint32_t myHalo = haloLoads / loaders;         // or one more
  if (myHalo >= 16) waitVmcnt<16>();
  else if (myHalo >= 8) waitVmcnt<8>();
  else waitVmcnt<0>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  half8 fb[C::STEPS][C::NC];
#pragma unroll
  for (int s = 0; s < C::STEPS; s++)
#pragma unroll
    for (int c = 0; c < C::NC; c++)
      fb[s][c] = *reinterpret_cast<const half8*>(smem + filter + (C::T * c + px) * 1152 + (s / C::PER_TAP) * 128 +
                                                 ((((s % C::PER_TAP) * (8 / C::PER_TAP) + part) ^ ((px >> 1) & 7)) << 4));

  // Most of it in accumulation registers, which an MFMA reads like the others: left to itself the compiler copies a third of the
  // fragments over in front of their MFMAs, tile by tile.
#pragma unroll
  for (int s = 0; s < C::STEPS; s++)
#pragma unroll
    for (int c = 0; c < C::NC; c++)
      if (s * C::NC + c < 48) asm volatile("" : "+a"(fb[s][c]));

  // Tile j of T rows: j = wave, wave + 4, ...
  // The rows of a finished tile go through LDS while the next one is multiplied, and out as whole lines, written through.
  const uint32_t tiles = (r1 - r0 + C::T - 1) / C::T, mine = (tiles + C::WAVES - 1 - wave) / C::WAVES;
  const uint32_t zeroPixel = haloPix * 128;
  // This lane's pixel of the tile: column and line of its image, and its place in the run.  The next tile is WAVES * T pixels on.
  uint32_t in = wave * C::T + px, ow, oh;
  {
    const uint32_t line = (r0 + in) / W;
    ow = r0 + in - line * W;
    oh = line % H;
  }
  const uint32_t lines = C::WAVES * C::T / W, columns = C::WAVES * C::T - lines * W, linesOn = lines % H;
  uint32_t tapMask = 0, first = 0;
  auto locate = [&] {
    uint32_t bits = r0 + in < r1 ? 0x1ffu : 0u;
    if (oh == 0) bits &= 0x1f8u;
    if (oh == H - 1) bits &= 0x03fu;
    if (ow == 0) bits &= 0x1b6u;
    if (ow == W - 1) bits &= 0x0dbu;
    tapMask = bits;
    first = min(in, R - 1);
    in += C::WAVES * C::T;
    ow += columns;
    oh += linesOn;
    if (ow >= W) { ow -= W; oh++; }
    if (oh >= H) oh -= H;
  };
  half8 fa[C::STEPS];
  auto readA = [&](int s) {
    const int tap = s / C::PER_TAP;
    const uint32_t pl = first + (uint32_t)(tap / 3) * W + tap % 3;
    const uint32_t at = (pl << 7) | ((part ^ ((pl >> 1) & 7)) << 4);
    const uint32_t inside = (uint32_t)__builtin_amdgcn_sbfe((int)tapMask, tap, 1);
    fa[s] = *reinterpret_cast<const half8*>(smem + (((at & inside) | (zeroPixel & ~inside)) ^ ((s % C::PER_TAP) * (128 / C::PER_TAP))));
  };
  if (!early && counts) waitVmcnt<1>();       // all but the count
  else waitVmcnt<0>();
  __builtin_amdgcn_s_waitcnt(0xc07f);       // lgkmcnt(0): the filter's place is free once everyone has read it
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  const GemmParams e = cusync::argumentsHere<GemmParams>();
  const __amdgpu_buffer_rsrc_t rD = makeRsrc(e.D, e.M * C::CHANNELS * 2);
  char* out = smem + filter + wave * C::OUT_BYTES;      // where the filter was
  floatx4 acc[C::NC], prev[C::NC];
  uint32_t prevRow = p.M;        // nothing to store before the first tile
#pragma unroll
  for (int c = 0; c < C::NC; c++) prev[c] = floatx4{};
  auto convert = [&](int c) {
    half4 o;
#pragma unroll
    for (int r = 0; r < 4; r++) o[r] = (half_t)applyEpilogue<EPILOGUE>(prev[c][r]);
    *reinterpret_cast<half4*>(out + px * C::OUT_PITCH + (C::T * c + 4 * part) * 2) = o;
  };
  uint4v rows[C::T / 8];
  auto gather = [&] {
#pragma unroll
    for (int s = 0; s < C::T / 8; s++) rows[s] = *reinterpret_cast<const uint4v*>(out + (s * 8 + lane / 8) * C::OUT_PITCH + (lane & 7) * 16);
  };
  auto store = [&] {
#pragma unroll
    for (int s = 0; s < C::T / 8; s++) {
      const uint32_t m = prevRow + s * 8 + lane / 8;
      __builtin_amdgcn_raw_buffer_store_b128(rows[s], rD, m < r1 ? (int)(m * 128 + (lane & 7) * 16) : (int)kOutOfRange, 0, 16 /* sc1 */);
    }
  };
  if (mine > 0) {
    locate();
#pragma unroll
    for (int s = 0; s < C::AHEAD; s++) readA(s);
    for (uint32_t k = 0; k < mine; k++) {
#pragma unroll
      for (int c = 0; c < C::NC; c++) acc[c] = floatx4{};
      staticFor<C::STEPS>([&](auto S) {
        constexpr int s = decltype(S)::value;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (s == C::STEPS - C::AHEAD) locate();
        readA((s + C::AHEAD) % C::STEPS);
#pragma unroll
        for (int c = 0; c < C::NC; c++) acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[s][c], fa[s], acc[c], 0, 0, 0);
        if constexpr (s < C::NC) convert(s);
        if constexpr (s == C::NC + 2) gather();
        if constexpr (s == C::NC + 6) store();
      });
#pragma unroll
      for (int c = 0; c < C::NC; c++) prev[c] = acc[c];
      prevRow = r0 + (wave + k * C::WAVES) * C::T;
      if (!early && k == 0 && tid == 0) stage.finishStart(startToken, p.launched, entered);
    }
#pragma unroll
    for (int c = 0; c < C::NC; c++) convert(c);
    gather(); store();
  }
  const unsigned long long tl2 = e.timeline ? wall_clock64() : 0;
  if (e.stage.isProducer()) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const uint32_t t0 = r0 / C::TILE_ROWS, touched = (r1 - 1) / C::TILE_ROWS - t0 + 1;
    if ((uint32_t)tid < touched) {
      const uint32_t t = t0 + tid, begin = t * C::TILE_ROWS, end = min(e.M, begin + C::TILE_ROWS);
      const uint32_t done = min(r1, end) - max(r0, begin);
      const uint32_t before = e.stage.releaseAll ? __hip_atomic_fetch_add(e.arrivals + t, done, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT)
                                                 : __hip_atomic_fetch_add(e.arrivals + t, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (before + done == end - begin) {
        dev::storeRelaxed(e.arrivals + t, 0);
        e.stage.countSeen();
        e.stage.raise(cusync_dim3{begin, 0, 0}, 1, true);
      }
    }
  }
  const cusync_dim3 t = {0, at, 0};
  if (tid == 0) recordTile(e, t, 0, tlEntry, tl0, tl1, tl2, e.timeline ? wall_clock64() : 0);
  e.stage.leave(e.launched);
}

}  // namespace gemm
}  // namespace cusync
