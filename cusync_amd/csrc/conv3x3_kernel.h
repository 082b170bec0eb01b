// 3x3, pad 1, stride 1 NHWC convolution whose input tile stays in LDS.
//
// The generic implicit-GEMM path (gemm_kernel_dma.h, kAConv) fetches every
// input pixel once per filter tap: nine trips through the vector memory path
// for data that is used nine times.  With stride 1 and pad 1 the output has the
// input's height and width, so in the flattened (n, h, w) pixel index the nine
// taps of output pixel m are input pixels m + (r-1)*W + (s-1): the 128 output
// pixels of a tile need the contiguous run of 128 + 2W + 2 input pixels around
// them.  That run (the tile plus its halo) is loaded into LDS once; the A
// fragment of tap (r, s) is then an LDS read at a shifted pixel index.  A lane
// whose tap falls outside the image (the flat neighbour would be a pixel of the
// next row or the next image) reads a pixel of zeros kept behind the run
// instead: one select on the address per tap, none on the fragments.  Only the
// filter is streamed, one 64-channel chunk of one tap per step, through a ring
// of stages as in the GEMM kernel; it is small and comes from L2 (a deeper ring
// measured the same: four and five stages against three on 28x28x128).
//
// LDS: [filter stages of BN x 64 halfs][halo: (BM + 2W + 2) pixels x C halfs][one pixel of zeros].
// An LDS read of 16 bytes per lane is served sixteen lanes at a time over all 64 banks, so the sixteen consecutive
// pixels (or filter rows) of such a group must fall into sixteen different places of 16 bytes.  A pixel's chunks are
// stored at chunk ^ (pixel & (C/8 - 1)); where a pixel is 128 bytes (C = 64), and in the filter's 128-byte rows, two
// neighbours cover all banks once and take one position: chunk ^ (pixel/2 & 7).  (With neighbours in different
// positions, rows r and r + 8 share their banks: pairs under RowSync 38.7 -> 37.6 us at 32x28x28x128, 51.5 -> 49.8 at
// 32x7x7x512, level at the other stages.  The 256x64 tile at 128 channels, which the chain takes only when told to, pays
// 2 to 4 % for the shift by nothing: one convolution 62.9 -> 65.6 us at 32x56x56x128.)
//
// Every wavefront (of a group) owns a 64 x 64 piece of the tile (two by two MFMA tiles), 32 x 64 of the 64-pixel tile: with
// 64 x 32 the kernel spent its time on LDS reads, three 16-byte reads per two
// MFMAs (measured: 0.54 us per 64-channel step against 0.1 us of MFMA work).
#pragma once

#include "gemm_kernel_dma.h"

namespace cusync {
namespace gemm {

// How many 16-channel products ahead of their use the fragments are read from LDS.  Measured on the ResNet pairs
// (56x56x64 / 28x28x128 / 14x14x256, stream-ordered, us): the compiler's own order 41.0 / 51.1 / 68.3; one ahead
// 39.9 / 48.6 / 63.8; two 39.7 / 49.4 / 65.2; the whole step up front 39.9 / 52.3 / 71.6.
constexpr int kFragsAhead = 1;

// How the accumulators leave a tile: as the kernel's wavefronts hold them, or (two groups, see KG) as they hold them
// once the groups have put their halves of the channels together.
//
// The runs of a tile leave it to the one that arrives last to add them up.  Adding up and storing a share each, as the
// k-slices of a GEMM do, makes every run wait for its siblings and the tile for two more round trips, and the sums it
// spreads are few (64 KB a run, not 200): pairs and chains of four, us, shared -> last arriver: 32x14x14x256 in two runs,
// pair under TileSync 51.3 -> 48.3, chain 94 -> 86; 12x14x14x256 in four runs, pair under RowSync 44.4 -> 39.9, chain under
// TileSync 82.7 -> 72.5; 2x14x14x256 in four 39.7 -> 39.0.  It is ahead at every batch of 14x14 and 28x28 images.
template<int BM_, int BN_, int WM_, int WN_, int THREADS_, int LDS_BYTES_>
struct HaloFinishCfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, THREADS = THREADS_, LDS_BYTES = LDS_BYTES_;
  static constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 32, TN = WTN / 32;
  static constexpr bool LAST_SLICE_ADDS = true;
};

// KG: groups of four wavefronts.  A tile that has its CU to itself (the halo of 128 channels and more fills the LDS)
// would run one wavefront per SIMD, which has nothing to issue while it waits for its fragments or at the barrier:
// a 64-channel step of the 128x128 tile took 0.57 us against 0.21 us of MFMAs.  Two groups share the tile: group g
// multiplies channels 32g..32g+31 of every step, the same 64 x 64 per wavefront and as many bytes read from LDS, and
// at the end each gives the other half of its sums through LDS.  Pairs under RowSync by the device's clock, one group ->
// two, in us: 8x28x28x128 32.7 -> 30.7, 8x14x14x256 39.2 -> 35.2, 32x14x14x256 48.5 -> 46.6, 8x7x7x512 39.1 -> 35.5,
// 32x7x7x512 54.6 -> 51.5; in one launch without runs 14x14x256 68.2 -> 56.3.  A step still takes 0.5 us: with the
// barrier between the two products and the first fragments of a step read ahead of it (a ring of four chunks where it
// fits) 48.3 at 32x14x14x256, and with tiles beginning at different steps of their range 47.2.
template<int BM_, int BN_, int WM_, int WN_, int STAGES_, int OCC_, int KG_ = 1>
struct Halo3x3Cfg {
  static constexpr int BM = BM_, BN = BN_, BK = 64, WM = WM_, WN = WN_, STAGES = STAGES_, OCC = OCC_, KG = KG_;
  static constexpr int WAVES = 4 * KG, THREADS = WAVES * 64;
  static constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 32, TN = WTN / 32, KS = BK / 16 / KG;      // KS: 16-channel products per wavefront and step
  static constexpr int B_ROW_BYTES = BK * 2, B_CPR = B_ROW_BYTES / 16;
  static constexpr int B_STAGE = BN * B_ROW_BYTES, B_LOADS = B_STAGE / 1024 / WAVES;
  static constexpr int B_BYTES = STAGES * B_STAGE;
  // The halves of two groups: of the wavefront's two rows of MFMA tiles, or of its two columns where it has one row.
  static constexpr bool HALVE_ROWS = TM == 2;
  static constexpr int EXCHANGE_BYTES = KG == 1 ? 0 : BM * BN * 4;
  // what the epilogue may use (finishTile): with two groups, whose wavefronts store twice as many rows at a time, also
  // some of the halo's place
  static constexpr int FINISH_BYTES = KG == 1 ? B_BYTES : (BM * (BN * 2 + 16) + 1023) / 1024 * 1024;
  using Finish = HaloFinishCfg<BM, BN, KG == 2 && HALVE_ROWS ? 2 * WM : WM, KG == 2 && !HALVE_ROWS ? 2 * WN : WN, THREADS, FINISH_BYTES>;
  static_assert(WM * WN == 4 && B_CPR == 8 && B_LOADS >= 1, "four wavefronts per group, 64-channel filter chunks");
  static_assert(KG == 1 || (KG == 2 && (TM == 2 || (TM == 1 && TN == 2))), "two groups exchange halves of a wavefront's tile");
  // Bytes of LDS a launch needs for images of width W with C channels.
  static uint32_t ldsBytes(uint32_t W, uint32_t C) {
    const uint32_t haloBytes = (BM + 2 * W + 3) * C * 2;      // the run of input pixels and one pixel of zeros behind it
    const uint32_t bytes = B_BYTES + (haloBytes + 1023) / 1024 * 1024, finish = FINISH_BYTES > EXCHANGE_BYTES ? FINISH_BYTES : EXCHANGE_BYTES;
    return bytes > finish ? bytes : finish;
  }
};

// One layer: all tiles of stage p.stage that this workgroup draws.  SPLIT: the launch may cut the 9 * C/64 steps of
// a tile into p.splitK runs (grid z), each a workgroup's, whose partial sums are put together as the GEMM's k-slices
// are (finishTile); the layers whose tiles are fewer than half the CUs are run that way.  A kernel without it does
// not carry the exchange's code.
template<class C, bool SPLIT>
__device__ __forceinline__ void convHalo3x3Layer(const GemmParams& p, uint32_t from = 0) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  __shared__ uint32_t sTicket, sLast;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = C::KG == 1 ? 0 : wave >> 2, inGroup = wave & 3;
  const int wm = inGroup / C::WN, wn = inGroup % C::WN;
  const uint32_t hi = lane >> 5;
  const cusync::DynStage& stage = p.stage;

  const uint32_t Cc = p.cvC, W = p.cvW, H = p.cvH;
  const uint32_t pixBytes = Cc * 2, cprMask = Cc / 8 - 1;             // C is a power of two
  const uint32_t swzShift = Cc == 64 ? 1 : 0;
  const uint32_t pixShift = 31 - __builtin_clz(pixBytes);
  const uint32_t haloPix = C::BM + 2 * W + 2;
  const uint32_t haloLoads = ((haloPix + 1) * pixBytes + 1023) / 1024;       // 1 KiB pieces; pixel haloPix is the pixel of zeros
  const uint32_t zeroPixel = haloPix << pixShift;
  const uint32_t chunksPerTapLog = pixShift - 7, chunksPerTap = 1u << chunksPerTapLog, steps = 9 * chunksPerTap;
  const uint4v rA = rawRsrc(p.A, p.M * Cc * 2);
  const uint4v rB = rawRsrc(p.B, p.N * p.ldb * 2);
  const uint32_t ldsBase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const uint32_t ldsHalo = ldsBase + C::B_BYTES;
  const char* halo = smem + C::B_BYTES;

  // Filter stage: [BN rows = output channels][BK halfs], chunk c of row n at slot c ^ (n/2 & 7).
  uint32_t bLoadRow[C::B_LOADS], bLoadChunk[C::B_LOADS];
#pragma unroll
  for (int q = 0; q < C::B_LOADS; q++) {
    const uint32_t slot = (wave * C::B_LOADS + q) * 64 + lane;
    bLoadRow[q] = slot / C::B_CPR;
    bLoadChunk[q] = (slot % C::B_CPR) ^ ((bLoadRow[q] >> 1) & 7);
  }
  // fragment of MFMA tile j, k-step kk: row wn*WTN + 32j + lane%32 (a multiple of 32 more does not change
  // row/2 & 7), chunk 2kk + hi
  uint32_t bFrag[C::KS];
  {
    const uint32_t row = wn * C::WTN + (lane & 31);
#pragma unroll
    for (int kk = 0; kk < C::KS; kk++) bFrag[kk] = row * C::B_ROW_BYTES + (((2 * (group * C::KS + kk) + hi) ^ ((row >> 1) & 7)) * 16);
  }

  const uint32_t numTiles = stage.numTiles();
  const bool consumer = stage.isConsumer();
  const uint32_t tmq = consumer ? stage.d.in.tileM : 1, tnq = consumer ? stage.d.in.tileN : 1;

  uint32_t dryXcds = 0, nextRaw = 0;
  const unsigned long long tlEntry = p.timeline ? wall_clock64() : 0;
  const unsigned long long entered = stage.enter();
  const uint32_t startToken = tid == 0 ? stage.beginStart() : 0;
  const bool noDraws = stage.noDraws;     // every tile is some workgroup's static first tile
  for (uint32_t round = 0;; round++) {
    const GemmParams p = cusync::argumentsHere<GemmParams>(from);
    const cusync::DynStage& stage = p.stage;
    if (tid == 0) sTicket = round == 0 ? stage.firstTicket(p.launched, dryXcds, noDraws) : stage.drawFinish(nextRaw, p.launched, round, dryXcds, noDraws);
    __syncthreads();
    const uint32_t ticket = sTicket;
    if (ticket >= numTiles) {
      if (tid == 0 && round == 0) stage.finishStart(startToken, p.launched, entered);
      break;
    }
    const cusync_dim3 t = stage.ticketToTile(ticket);
    const unsigned long long tl0 = p.timeline ? wall_clock64() : 0;
    const uint32_t m0 = t.y * C::BM, n0 = t.x * C::BN;
    // this workgroup's steps of the tile: all of them, or run t.z of p.kPerSlice / 64 steps
    const uint32_t itBegin = SPLIT ? min(steps, t.z * (p.kPerSlice / C::BK)) : 0;
    const uint32_t itEnd = SPLIT ? min(steps, itBegin + p.kPerSlice / C::BK) : steps;

    // Which of the nine taps of this lane's output pixels lie inside the image: bit 3r + s.
    uint32_t tapMask[C::TM];
#pragma unroll
    for (int i = 0; i < C::TM; i++) {
      const uint32_t m = m0 + wm * C::WTM + i * 32 + (lane & 31);
      const uint32_t ow = m % W, oh = (m / W) % H;
      uint32_t bits = 0;
#pragma unroll
      for (uint32_t r = 0; r < 3; r++)
#pragma unroll
        for (uint32_t s = 0; s < 3; s++)
          if (oh + r >= 1 && oh + r <= H && ow + s >= 1 && ow + s <= W) bits |= 1u << (3 * r + s);
      tapMask[i] = m < p.M ? bits : 0;
    }

    // A consumer waits for every producer row block the halo reaches, once per producer channel tile
    // (every wave for itself: each one fetches part of the halo).
    if (consumer) {
      const uint32_t lo = m0 > W + 1 ? m0 - (W + 1) : 0, hiRow = min(m0 + C::BM + W, p.M - 1);
      if (stage.d.in.kind == CUSYNC_POLICY_ROWSYNC) {
        stage.waitWaveRows(lo, hiRow, tmq, 0, 1);
      } else {
        const uint32_t perTile = stage.d.in.kind == CUSYNC_POLICY_CONV2DTILESYNC ? 9 * tnq : tnq;
        for (uint32_t ct = 0; ct < Cc / tnq; ct++)
          stage.waitWaveRows(lo, hiRow, tmq, ct * perTile, 0);
      }
    }

    // Halo: input pixels m0 - (W+1) .. m0 + BM + W, 1 KiB per load; pixels before the first or after the
    // last image are sent out of range and arrive as zeros.
    for (uint32_t q = wave; q < haloLoads; q += C::WAVES) {
      const uint32_t byteOff = q * 1024 + lane * 16;
      const uint32_t pl = byteOff >> pixShift, slot = (byteOff & (pixBytes - 1)) >> 4;
      const uint32_t chunk = slot ^ ((pl >> swzShift) & cprMask);
      const uint32_t flat = m0 + pl - (W + 1);                       // wraps below zero for the first tile
      const bool inside = m0 + pl >= W + 1 && flat < p.M && pl < haloPix;
      loadToLds(rA, __builtin_amdgcn_readfirstlane(ldsHalo + q * 1024), inside ? (flat * Cc + chunk * 8) * 2 : kOutOfRange);
    }
    // Filter chunk `it` (tap it / chunksPerTap, channels (it % chunksPerTap) * 64 ..) into stage (it - itBegin) % STAGES.
    auto issueB = [&](uint32_t it) {
      const uint32_t lds = ldsBase + ((it - itBegin) % C::STAGES) * C::B_STAGE + wave * C::B_LOADS * 1024;
#pragma unroll
      for (int q = 0; q < C::B_LOADS; q++) {
        const bool live = it < itEnd && n0 + bLoadRow[q] < p.N;
        loadToLds(rB, __builtin_amdgcn_readfirstlane(lds + q * 1024),
                  live ? ((n0 + bLoadRow[q]) * p.ldb + it * C::BK + bLoadChunk[q] * 8) * 2 : kOutOfRange);
      }
    };
#pragma unroll
    for (uint32_t it = 0; it < C::STAGES - 1; it++) issueB(itBegin + it);
    if (tid == 0 && round == 0) stage.finishStart(startToken, p.launched, entered);
    const unsigned long long tl1 = p.timeline ? wall_clock64() : 0;

    floatx16 acc[C::TM][C::TN];
#pragma unroll
    for (int i = 0; i < C::TM; i++)
#pragma unroll
      for (int j = 0; j < C::TN; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    const uint32_t aPixel0 = wm * C::WTM + (lane & 31) + W + 1;       // this lane's first output pixel inside the halo
    for (uint32_t it = itBegin; it < itEnd; it++) {
      waitVmcnt<(C::STAGES - 2) * C::B_LOADS>();     // chunk `it` (and, the first time, the halo) has landed
      __builtin_amdgcn_s_barrier();                   // ... for everyone; everyone is done with chunk it-1
      asm volatile("" ::: "memory");
      issueB(it + C::STAGES - 1);
      const uint32_t tap = it >> chunksPerTapLog, cc = it & (chunksPerTap - 1);
      const int32_t shift = ((int32_t)(tap / 3) - 1) * (int32_t)W + (int32_t)(tap % 3) - 1;
      const char* sb = smem + ((it - itBegin) % C::STAGES) * C::B_STAGE;
      uint32_t aBase[C::TM], aSwz[C::TM];
#pragma unroll
      for (int i = 0; i < C::TM; i++) {
        const uint32_t pl = (uint32_t)((int32_t)(aPixel0 + i * 32) + shift);
        aBase[i] = (tapMask[i] >> tap) & 1 ? pl << pixShift : zeroPixel;
        aSwz[i] = (pl >> swzShift) & cprMask;      // any slot of the pixel of zeros will do
      }
      // The fragments of 16 channels are requested kFragsAhead products of 16 channels before they are used.
      half8 fb[C::KS][C::TN], fa[C::KS][C::TM];
      auto readFrags = [&](int kk) {
#pragma unroll
        for (int j = 0; j < C::TN; j++) fb[kk][j] = *reinterpret_cast<const half8*>(sb + bFrag[kk] + j * 32 * C::B_ROW_BYTES);
#pragma unroll
        for (int i = 0; i < C::TM; i++) {
          const uint32_t chunk = cc * (C::BK / 8) + 2 * (group * C::KS + kk) + hi;
          fa[kk][i] = *reinterpret_cast<const half8*>(halo + aBase[i] + ((chunk ^ aSwz[i]) << 4));
        }
      };
#pragma unroll
      for (int kk = 0; kk < kFragsAhead && kk < C::KS; kk++) readFrags(kk);
#pragma unroll
      for (int kk = 0; kk < C::KS; kk++) {
        __builtin_amdgcn_sched_barrier(0);      // left alone, the compiler issues each read two MFMAs before its use
        if (kk + kFragsAhead < C::KS) readFrags(kk + kFragsAhead);
#pragma unroll
        for (int i = 0; i < C::TM; i++)
#pragma unroll
          for (int j = 0; j < C::TN; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[kk][j], fa[kk][i], acc[i][j], 0, 0, 0);
      }
    }

    // The loads issued for chunks past the last one (zeros) may still be on their way into LDS, which the
    // epilogue is about to reuse.
    waitVmcnt<0>();
    const unsigned long long tl2 = p.timeline ? wall_clock64() : 0;
    const GemmParams e = cusync::argumentsHere<GemmParams>(from);
    if (tid == 0) nextRaw = e.stage.drawBegin(dryXcds, noDraws);     // settled after the epilogue
    using F = typename C::Finish;
    bool completed;
    if constexpr (C::KG == 1) {
      completed = finishTile<F, SPLIT>(e, acc, t, wm, wn, lane, &sLast, smem);
    } else {
      // Group g keeps half g of the sums, its own and the other group's: sixteen bytes per lane and piece, every
      // lane's values in a place of their own.
      floatx16 sums[F::TM][F::TN];
      constexpr int HALF = F::TM * F::TN;
      static_assert(F::TM == 1, "half of two rows, or one of two columns, of MFMA tiles");
      auto place = [&](int to, int h, int g) { return smem + (((inGroup * 2 + to) * HALF + h) * 4 + g) * 1024 + lane * 16; };
      auto part = [&](int half, int h) { return C::HALVE_ROWS ? acc[half][h] : acc[0][half]; };
      __syncthreads();             // every wavefront is out of the steps and its loads have landed
#pragma unroll
      for (int h = 0; h < HALF; h++) {
        floatx16 give;
        if (group == 0) { give = part(1, h); sums[0][h] = part(0, h); }
        else { give = part(0, h); sums[0][h] = part(1, h); }
#pragma unroll
        for (int g = 0; g < 4; g++)
          *reinterpret_cast<floatx4*>(place(1 - group, h, g)) = floatx4{give[4 * g], give[4 * g + 1], give[4 * g + 2], give[4 * g + 3]};
      }
      __syncthreads();
#pragma unroll
      for (int h = 0; h < HALF; h++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const floatx4 v = *reinterpret_cast<const floatx4*>(place(group, h, g));
#pragma unroll
          for (int e = 0; e < 4; e++) sums[0][h][4 * g + e] += v[e];
        }
      if constexpr (C::HALVE_ROWS) completed = finishTile<F, SPLIT>(e, sums, t, 2 * wm + group, wn, lane, &sLast, smem);
      else completed = finishTile<F, SPLIT>(e, sums, t, wm, 2 * wn + group, lane, &sLast, smem);
    }
    cusync_dim3 done = {m0, n0, 0};
    if (completed && e.stage.isProducer()) e.stage.post(done, 1, e.stage.storesThrough());
    else __syncthreads();
    if (tid == 0) recordTile(e, t, round, tlEntry, tl0, tl1, tl2, e.timeline ? wall_clock64() : 0);
  }
  const GemmParams atEnd = cusync::argumentsHere<GemmParams>(from);
  atEnd.stage.leave(atEnd.launched);
}

template<class C, bool SPLIT = false>
__global__ __launch_bounds__(C::THREADS, C::OCC) void convHalo3x3Kernel(GemmParams p) {
  convHalo3x3Layer<C, SPLIT>(p);
}

// A chain of layers in ONE launch: every workgroup works through the tiles of layer 0 it can draw, then those
// of layer 1, and so on; a tile of layer l+1 waits on the semaphores of layer l exactly as it does when the
// layers are separate launches.  No wait kernel and no second launch sit between a producer and its consumer
// (on this device the first dispatch on another stream starts 15-20 us after the producer did, about as long
// as a whole 3x3 layer of the ResNet shapes takes).  Forward progress: the launch has no more workgroups than
// stay resident, and a workgroup only moves on to layer l+1 when layer l has no tile left to hand out, so every
// tile a consumer tile waits for is already in the hands of a running workgroup.
constexpr int kMaxFusedLayers = 8;
struct ConvChainParams {
  GemmParams layer[kMaxFusedLayers];
  uint32_t layers;
};

template<class C>
__global__ __launch_bounds__(C::THREADS, C::OCC) void convHalo3x3ChainKernel(ConvChainParams cp) {
  for (uint32_t l = 0; l < cp.layers; l++) {
    convHalo3x3Layer<C, false>(cp.layer[l], l * sizeof(GemmParams));
    __syncthreads();        // everyone has read the last ticket of this layer before the next one's is written
  }
}

}  // namespace gemm
}  // namespace cusync
