// 3x3, pad 1, stride 1 convolution for layers whose tiles are few: 64 output channels to a workgroup, the channels of the
// sum divided among its wavefronts.
//
// The input tile and its halo lie in LDS as in conv3x3_kernel.h.  There four wavefronts share every 64-channel step of the
// filter: a barrier and a wait for the ring of stages per step, 0.5 us against 0.2 us of MFMAs, and tiles too few for the
// device have their steps cut into runs whose sums go through memory.  Here a wavefront takes whole units (64 channels of one
// tap) by itself, every fourth one: BM x 64 outputs in its accumulators, a ring of its own for its units' filter rows, no
// barrier between the halo's arrival and the end.  The four partial sums come together through LDS, a quarter of the tile per
// wavefront.  A fragment read from LDS is used twice (halo) or TM times (filter): 6 reads per 8 MFMAs of the 128-row tile,
// where 64 x 64 per wavefront takes 8.
//
// Pairs, us, tiles in runs -> this kernel, under RowSync: 32x14x14x256 49.1 -> 37.3, under TileSync 49.5 -> 38.1 (a layer's loop 10.3
// -> 8.2, start to first load 2.0 -> 0.3, exchange and store 4.5 -> 2.2); 8x14x14x256 39.4 -> 27.0; 32x7x7x512 51.3 -> 42.6; 8x28x28x128
// 35.2 -> 24.7; 1x28x28x128 33.6 -> 22.0.  Chains of four: 32x14x14x256 85.3 -> 65.4, 1x14x14x256 67.7 -> 45.6, 32x7x7x512 89.9 -> 76.4.  What bounds it at 32x14x14x256: MFMAs alone on as many CUs take 5.8 us a layer (1.95 GHz
// on such data), the loop 7.7 without its direct loads; at 512 channels the filter: 590 KB per workgroup at 53 bytes/ns.
//
// A workgroup has one tile and the launch a workgroup for each (soloTileFor): with a loop over tiles around it the compiler
// worked out a thousand instructions ahead of the first one, 2 us.  The arguments it needs are read in one go at the top:
// each group of scalar loads behind a branch is another round trip.
#pragma once

#include "conv3x3_kernel.h"

namespace cusync {
namespace gemm {

// RING: stages of a wavefront's ring, one unit each.
template<int BM_, int RING_, int OCC_>
struct HaloSoloCfg {
  static constexpr int BM = BM_, BN = 64, BK = 64, RING = RING_, OCC = OCC_;
  static constexpr int KG = 4, THREADS = KG * 64;
  static constexpr int TM = BM / 32, TN = BN / 32, PER = TM * TN / KG;      // MFMA tiles of a wavefront, and how many of them it puts together at the end
  static constexpr int STAGE = BN * BK * 2, LOADS = STAGE / 1024, RING_BYTES = KG * RING * STAGE;
  static constexpr int EXCHANGE_BYTES = KG * (KG - 1) * PER * 4096;
  static constexpr int FINISH_WM = TM == 4 ? 4 : 2, FINISH_WN = KG / FINISH_WM;
  using Finish = HaloFinishCfg<BM, BN, FINISH_WM, FINISH_WN, THREADS, RING_BYTES>;
  static_assert((TM == 4 || TM == 2) && TN == 2 && RING == 2, "the loop's waits and the exchange are for these");
  static uint32_t ldsBytes(uint32_t W, uint32_t C) {
    const uint32_t haloBytes = (BM + 2 * W + 3) * C * 2;
    const uint32_t bytes = RING_BYTES + (haloBytes + 1023) / 1024 * 1024;
    return bytes > EXCHANGE_BYTES ? bytes : EXCHANGE_BYTES;
  }
};

// The 128 columns of a tile are two workgroups' (half 0 and 1 of grid z).  SPLIT: grid z is 2 * runs, and each half's units are
// cut into that many runs (a power of two), a workgroup each; the run that arrives last adds the halves' partial sums up in the
// order of the runs.  Counters per tile, 0 between launches: arrivals of half h in the lower 16 bits of counter h, finished halves
// in the upper 16 bits of counter 0; all changes are additions, so neither disturbs the other.
template<class C, bool SPLIT>
__device__ __forceinline__ void convHaloSoloTile(const GemmParams& p) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  __shared__ uint32_t sLast;

  asm volatile("" :: "s"(p.cvC), "s"(p.cvW), "s"(p.cvH), "s"(p.A), "s"(p.B), "s"(p.M), "s"(p.N), "s"(p.ldb), "s"(p.launched), "s"(p.splitK), "s"(p.timeline));
  asm volatile("" :: "s"(p.stage.d.grid.x), "s"(p.stage.d.grid.y), "s"(p.stage.d.grid.z), "s"(p.stage.d.flags), "s"(p.stage.d.opts), "s"(p.stage.d.in.kind), "s"(p.stage.d.out.kind), "s"(p.stage.d.startCounter), "s"((uint32_t)p.stage.noDraws));
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t hi = lane >> 5;
  const cusync::DynStage& stage = p.stage;

  const uint32_t Cc = p.cvC, W = p.cvW, H = p.cvH;
  const uint32_t pixBytes = Cc * 2, cprMask = Cc / 8 - 1;             // C is a power of two
  const uint32_t swzShift = Cc == 64 ? 1 : 0;
  const uint32_t pixShift = 31 - __builtin_clz(pixBytes);
  const uint32_t haloPix = C::BM + 2 * W + 2;
  const uint32_t haloLoads = ((haloPix + 1) * pixBytes + 1023) / 1024;
  const uint32_t chunksPerTapLog = pixShift - 7, chunksPerTap = 1u << chunksPerTapLog, units = 9 * chunksPerTap;
  const uint4v rA = rawRsrc(p.A, p.M * Cc * 2);
  const uint4v rB = rawRsrc(p.B, p.N * p.ldb * 2);
  const uint32_t ldsBase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const uint32_t ldsHalo = ldsBase + C::RING_BYTES;
  const uint32_t ring = wave * (C::RING * C::STAGE);
  const uint32_t zeroPixel = C::RING_BYTES + (haloPix << pixShift);

  const bool consumer = stage.isConsumer();
  const uint32_t tmq = consumer ? stage.d.in.tileM : 1, tnq = consumer ? stage.d.in.tileN : 1;

  const unsigned long long tlEntry = p.timeline ? wall_clock64() : 0;
  const unsigned long long entered = stage.enter();
  // What a wavefront loads behind the start count arrives behind it, 1 to 3 us when hundreds of workgroups count at once: the one
  // that counts leaves the halo to the others.
  const bool counts = stage.countsStart();
  const uint32_t loaders = counts ? C::KG - 1 : C::KG, loader = counts ? wave - 1 : wave;       // (all ones where it has nothing to load)
  const uint32_t startToken = tid == 0 ? stage.beginStart() : 0;
  cusync_dim3 t;
  if (stage.noDraws && (stage.d.flags & CUSYNC_STAGE_IDENTITY_ORDER)) t = deal::evenTile(stage.d.grid, p.launched, blockIdx.x);
  else t = stage.ticketToTile(blockIdx.x);
  const unsigned long long tl0 = p.timeline ? wall_clock64() : 0;
  const uint32_t runsLog = SPLIT ? (uint32_t)__builtin_ctz(p.splitK) - 1 : 0, half = SPLIT ? t.z >> runsLog : t.z, run = SPLIT ? t.z & ((1u << runsLog) - 1) : 0;
  const uint32_t m0 = t.y * C::BM, n0 = (t.x * 2 + half) * C::BN;
  const uint32_t perRun = SPLIT ? (units + (1u << runsLog) - 1) >> runsLog : units, first = run * perRun + wave;
  const uint32_t mine = SPLIT ? (run * perRun < units ? min(perRun, units - run * perRun) : 0u) : units;
  const uint32_t myUnits = (mine + C::KG - 1 - wave) / C::KG;

  // Filter stage: [64 rows = output channels][64 halfs], chunk c of row n at slot c ^ (n/2 & 7); a load is eight rows.
  uint32_t bOff[2];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const uint32_t row = q * 8 + lane / 8;
    bOff[q] = ((n0 + row) * p.ldb + (((uint32_t)(lane % 8) ^ ((row >> 1) & 7)) * 8)) * 2;
  }
  auto issueB = [&](uint32_t u, int q) {
    const uint32_t unit = first + C::KG * u;
    const uint32_t add = u < myUnits ? unit * (C::BK * 2) + (uint32_t)(q / 2) * 16 * p.ldb * 2 : kOutOfRange;
    loadToLds(rB, __builtin_amdgcn_readfirstlane(ldsBase + ring + (u & 1) * C::STAGE + q * 1024), bOff[q & 1] + add);
  };

  // A producer of nothing it reads has its weights from the start; a consumer reads them ahead of its wait only where it may.
  const bool weightsFirst = !consumer || (stage.d.opts & CUSYNC_OPT_REORDER_TILE_LOADS);
  auto issueStage = [&](uint32_t u) {
#pragma unroll
    for (int q = 0; q < C::LOADS; q++) issueB(u, q);
  };
  if (weightsFirst) issueStage(0);
  if (weightsFirst && consumer) issueStage(1);
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
  // Halo, as in conv3x3_kernel.h.
  for (uint32_t q = loader; q < haloLoads; q += loaders) {
    const uint32_t byteOff = q * 1024 + lane * 16;
    const uint32_t pl = byteOff >> pixShift, slot = (byteOff & (pixBytes - 1)) >> 4;
    const uint32_t chunk = slot ^ ((pl >> swzShift) & cprMask);
    const uint32_t flat = m0 + pl - (W + 1);
    const bool inside = m0 + pl >= W + 1 && flat < p.M && pl < haloPix;
    loadToLds(rA, __builtin_amdgcn_readfirstlane(ldsHalo + q * 1024), inside ? (flat * Cc + chunk * 8) * 2 : kOutOfRange);
  }
  if (!weightsFirst) issueStage(0);
  if (!weightsFirst || !consumer) issueStage(1);
  if (tid == 0) stage.finishStart(startToken, p.launched, entered);
  const unsigned long long tl1 = p.timeline ? wall_clock64() : 0;

  // Which of the nine taps of this lane's output pixels lie inside the image: bit 3r + s.
  uint32_t tapMask[C::TM];
#pragma unroll
  for (int i = 0; i < C::TM; i++) {
    const uint32_t m = m0 + i * 32 + (lane & 31);
    const uint32_t line = m / W, ow = m - line * W, oh = line % H;
    uint32_t bits = m < p.M ? 0x1ffu : 0u;
    if (oh == 0) bits &= 0x1f8u;
    if (oh == H - 1) bits &= 0x03fu;
    if (ow == 0) bits &= 0x1b6u;
    if (ow == W - 1) bits &= 0x0dbu;
    tapMask[i] = bits;
    asm volatile("" : "+v"(tapMask[i]));
  }

  floatx16 acc[C::TM][C::TN];
#pragma unroll
  for (int i = 0; i < C::TM; i++)
#pragma unroll
    for (int j = 0; j < C::TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

  const uint32_t aPixel0 = (lane & 31) + W + 1;
  const uint32_t bAddr0 = ring + (lane & 31) * 128 + ((hi ^ ((lane >> 1) & 7)) << 4);
  // LDS addresses of this lane's pixels for unit u, first 16 channels; product kk of the unit is at the address ^ 32 kk.
  uint32_t aAddr[C::TM];
  auto locate = [&](uint32_t u) {
    const uint32_t unit = min(first + C::KG * u, units - 1);
    const uint32_t tap = unit >> chunksPerTapLog, cc = unit & (chunksPerTap - 1);
    const int32_t shift = ((int32_t)(tap / 3) - 1) * (int32_t)W + (int32_t)(tap % 3) - 1;
#pragma unroll
    for (int i = 0; i < C::TM; i++) {
      const uint32_t pl = (uint32_t)((int32_t)(aPixel0 + i * 32) + shift);
      const uint32_t at = C::RING_BYTES + (pl << pixShift) + (((cc * 8 + hi) ^ ((pl >> swzShift) & cprMask)) << 4);
      const uint32_t inside = (uint32_t)__builtin_amdgcn_sbfe((int)tapMask[i], tap, 1);
      aAddr[i] = (at & inside) | (zeroPixel & ~inside);
    }
  };
  half8 fa[4][C::TM], fb[4][C::TN];
  auto readA = [&](int kk, int i) { fa[kk][i] = *reinterpret_cast<const half8*>(smem + (aAddr[i] ^ (kk << 5))); };
  auto readB = [&](uint32_t u, int kk, int j) {
    fb[kk][j] = *reinterpret_cast<const half8*>(smem + ((bAddr0 + (u & 1) * C::STAGE) ^ (kk << 5)) + j * 4096);
  };

  if (weightsFirst && consumer) waitVmcnt<0>();
  else waitVmcnt<C::LOADS>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);       // lgkmcnt(0): with scalar loads under way here the compiler would wait for everything at the loop's head
  locate(0);
  // Fragments are read two products (filter) and three (halo) ahead of their MFMAs, in the place between two MFMAs each; a unit's
  // loads go out while its last product runs, into the stage whose fragments have just been read.
  // (The first ones in the loop's order, which the compiler's counts of outstanding reads at the loop's head go by)
#pragma unroll
  for (int kk = 0; kk < 3; kk++) {
    if (kk > 0) {
#pragma unroll
      for (int j = 0; j < C::TN; j++) { readB(0, kk - 1, j); __builtin_amdgcn_sched_barrier(0); }
    }
#pragma unroll
    for (int i = 0; i < C::TM; i++) { readA(kk, i); __builtin_amdgcn_sched_barrier(0); }
  }
  for (uint32_t u = 0; u < myUnits; u++) {
    staticFor<4>([&](auto K) {
      constexpr int kk = decltype(K)::value;
      constexpr int T = C::TM * C::TN;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (kk == 1) locate(u + 1);
      if constexpr (kk == 2) waitVmcnt<0>();          // stage u + 1
      if constexpr (kk == 3) asm volatile("s_waitcnt lgkmcnt(%0)" :: "n"(C::TM + C::TN) : "memory");      // stage u's last fragments are here: its place is free
#pragma unroll
      for (int m = 0; m < T; m++) {
        const int i = m / C::TN, j = m % C::TN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[kk][j], fa[kk][i], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (m < C::TN) readB(kk < 2 ? u : u + 1, (kk + 2) & 3, m);
        else if (m < C::TN + C::TM) readA((kk + 3) & 3, m - C::TN);
        if constexpr (kk == 3) {
#pragma unroll
          for (int q = 0; q < C::LOADS / T; q++) issueB(u + 2, m * (C::LOADS / T) + q);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    });
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  waitVmcnt<0>();
  const unsigned long long tl2 = p.timeline ? wall_clock64() : 0;
  const GemmParams e = cusync::argumentsHere<GemmParams>();

  using F = typename C::Finish;
  floatx16 sums[F::TM][F::TN];
  static_assert(F::TM == 1 && F::TN == C::PER, "");
  auto place = [&](uint32_t owner, uint32_t giver, int h, int g) {
    return smem + (((owner * (C::KG - 1) + giver) * C::PER + h) * 4 + g) * 1024 + lane * 16;
  };
  __syncthreads();
#pragma unroll
  for (int o = 0; o < C::KG; o++) {
#pragma unroll
    for (int h = 0; h < C::PER; h++) {
      const floatx16& v = acc[(o * C::PER + h) / C::TN][(o * C::PER + h) % C::TN];
      if (o == wave) sums[0][h] = v;
      else {
#pragma unroll
        for (int g = 0; g < 4; g++)
          *reinterpret_cast<floatx4*>(place(o, wave < o ? wave : wave - 1, h, g)) = floatx4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < C::KG - 1; s++)
#pragma unroll
    for (int h = 0; h < C::PER; h++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const floatx4 v = *reinterpret_cast<const floatx4*>(place(wave, s, h, g));
#pragma unroll
        for (int r = 0; r < 4; r++) sums[0][h][4 * g + r] += v[r];
      }
  uint32_t* halves = e.arrivals + 2 * (t.y * e.stage.d.grid.x + t.x);
  if constexpr (SPLIT) {
    const uint32_t runs = 1u << runsLog;
    const __amdgpu_buffer_rsrc_t rPart = makeRsrc(e.partials, e.partialBytes);
    const uint32_t tileBase = ((t.y * e.stage.d.grid.x + t.x) * 2 + half) * runs;
    auto at = [&](uint32_t z, int h, int g) { return (int)((tileBase + z) * (C::BM * C::BN * 4) + (((wave * C::PER + h) * 4 + g) * 64 + lane) * 16); };
#pragma unroll
    for (int h = 0; h < C::PER; h++)
#pragma unroll
      for (int g = 0; g < 4; g++)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, floatx4{sums[0][h][4 * g], sums[0][h][4 * g + 1], sums[0][h][4 * g + 2], sums[0][h][4 * g + 3]}),
                                               rPart, at(run, h, g), 0, 16 /* sc1 */);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      const uint32_t before = e.stage.countIn(halves + half) & 0xffffu;
      const bool last = before == runs - 1;
      if (last) { __hip_atomic_fetch_sub(halves + half, runs, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); e.stage.countSeen(); }
      sLast = last;
    }
    __syncthreads();
    if (!sLast) {
      if (tid == 0) recordTile(e, t, 0, tlEntry, tl0, tl1, tl2, e.timeline ? wall_clock64() : 0);
      e.stage.leave(e.launched);
      return;
    }
    for (uint32_t z = 0; z < runs; z++) {
      floatx4 v[C::PER][4];
#pragma unroll
      for (int h = 0; h < C::PER; h++)
#pragma unroll
        for (int g = 0; g < 4; g++) v[h][g] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rPart, at(z, h, g), 0, 16 /* sc1 */));
#pragma unroll
      for (int h = 0; h < C::PER; h++)
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
          for (int r = 0; r < 4; r++) sums[0][h][4 * g + r] = z == 0 ? v[h][g][r] : sums[0][h][4 * g + r] + v[h][g][r];
    }
  }
  const cusync_dim3 part = {t.x * 2 + half, t.y, 0};
  finishTile<F, false>(e, sums, part, wave / F::WN, wave % F::WN, lane, &sLast, smem);
  bool completed = false;
  if (e.stage.isProducer()) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      const uint32_t before = e.stage.releaseAll ? __hip_atomic_fetch_add(halves, 0x10000u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT)
                                                 : __hip_atomic_fetch_add(halves, 0x10000u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool last = before >> 16 == 1;
      if (last) { __hip_atomic_fetch_sub(halves, 0x20000u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); e.stage.countSeen(); }
      sLast = last;
    }
    __syncthreads();
    completed = sLast != 0;
  }
  cusync_dim3 done = {m0, t.x * 2 * C::BN, 0};
  if (completed) e.stage.post(done, 1, e.stage.storesThrough());
  else __syncthreads();
  if (tid == 0) recordTile(e, t, 0, tlEntry, tl0, tl1, tl2, e.timeline ? wall_clock64() : 0);
  e.stage.leave(e.launched);
}

template<class C, bool SPLIT>
__global__ __launch_bounds__(C::THREADS, C::OCC) void convHaloSoloKernel(GemmParams p) {
  convHaloSoloTile<C, SPLIT>(p);
}

}  // namespace gemm
}  // namespace cusync
