// The attention stage for up to 32 query rows whose key range is split over workgroups: decoding, a few new rows
// behind a long key/value cache.
//
// attentionKernel gives each of a workgroup's four wavefronts 32 query rows; with no more than 32 rows in all three of
// them have nothing to do, and a block of 64 keys takes the fourth 1.6 us, one after the other.  Here the four
// wavefronts share the query rows and divide the keys: 32 keys (16 KB of K and V) at a time, wavefront w taking the
// pieces w, w + 4, ... of the workgroup's range.  Every wavefront loads what it works on into a ring of two pieces of
// its own, so the loop over the keys has no barrier.  The cached rows are nobody's product: their first pieces are
// under way before the projection that makes the queries is waited for.
//
// What bounds it is latency: K and V of 2064 rows and 12 heads are 12.7 MB, two microseconds of memory; a split's share
// goes out, is counted and comes back in three round trips (5 us), and a wavefront's piece takes 0.9 us.  Measured with
// the chain's own splits, 12 heads, launch boundary included: 16 rows behind 2048 19.6 us (25.8 with attentionKernel in
// the same splits, 35.6 in the two that it used to be given), behind 8192 25.8 (95 in two).
//
// The four running results are put together through LDS, wavefront w taking head-dim 32 w .. 32 w + 31 from there on
// (also when the split that arrives last puts the splits together: all of a tile's shares are read by four wavefronts
// at once, eight splits per round trip).  The sums go in wavefront order and in split order.
#pragma once

#include "attention_kernel.h"

namespace cusync {
namespace attn {

constexpr int kFewRows = 32;
constexpr int kPieceKeys = 32, kPieceBytes = 2 * kPieceKeys * kRowBytes, kPieceLoads = kPieceBytes / 1024;
constexpr int kFewLdsBytes = 4 * 2 * kPieceBytes;

__global__ __launch_bounds__(kThreads, 1) void attentionFewKernel(AttnParams p) {
  constexpr uint32_t from = 0;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  __shared__ uint32_t sTicket, sLast;
  __shared__ float sStat[2][4][64];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t hi = lane >> 5;
  const cusync::DynStage& stage = p.stage;
  const uint32_t E = p.heads * kHD;
  const uint32_t total = p.cached + p.S;
  const uint32_t bufBytes = total * p.ldq * 2;
  const uint4v rLds = rawRsrc(p.qkv, bufBytes);
  const __amdgpu_buffer_rsrc_t rReg = makeRsrc(p.qkv, bufBytes);
  char* ring = smem + wave * 2 * kPieceBytes;
  const uint32_t ringLds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring;

  // Layout and fragments of K and V as in attentionKernel, with 32 rows to a piece: load q fills rows 4q + lane/16.
  const uint32_t ldRow = lane >> 4;
  const uint32_t vChunk = (lane & 15) ^ (4 * ((lane >> 4) & 1));
  uint32_t kFrag[8];
#pragma unroll
  for (int s = 0; s < 8; s++) kFrag[s] = (lane & 31) * kRowBytes + (((2 * s + hi) ^ (lane & 15)) * 16);
  const uint32_t flip = (lane >> 2) & 1;
  const uint32_t vRowOff = (4 * hi + ((lane & 15) >> 2)) * kRowBytes;
  const uint32_t vColOff = (2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) * 16 + (lane & 1) * 8;
  const uint32_t vEven = vRowOff + vColOff + 64 * flip, vOdd = vRowOff + vColOff + 64 - 64 * flip;

  const uint32_t numTiles = stage.numTiles();
  const bool consumer = stage.isConsumer();
  const uint32_t tmq = consumer ? stage.d.in.tileM : 1, tnq = consumer ? stage.d.in.tileN : 1;
  const uint32_t zWait = consumer && (stage.d.in.kind == CUSYNC_POLICY_ROWSYNC || stage.d.in.kind == CUSYNC_POLICY_CONSECUTIVESYNC) ? 1 : 0;
  // the producer's tiles of all query rows (its only rows) under columns col .. col + kHD - 1
  auto waitRows = [&](uint32_t col) {
    for (uint32_t c = col / tnq * tnq; c < col + kHD; c += tnq) {
      stage.waitWaveRows(0, p.S - 1, tmq, c, zWait);
      if (zWait) break;
    }
  };

  uint32_t dryXcds = 0, nextRaw = 0;
  const unsigned long long tlEntry = p.timeline ? wall_clock64() : 0;
  const unsigned long long entered = stage.enter();
  const uint32_t startToken = tid == 0 ? stage.beginStart() : 0;
  const bool noDraws = stage.noDraws;
  for (uint32_t round = 0;; round++) {
    const AttnParams p = cusync::argumentsHere<AttnParams>(from);
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
    const uint32_t head = t.x;
    const uint32_t pieces = (total + kPieceKeys - 1) / kPieceKeys, perSplit = p.chunk * (kBKV / kPieceKeys);
    const uint32_t splits = (pieces + perSplit - 1) / perSplit;       // = grid z: every split has keys
    const uint32_t first = t.z * perSplit + wave, end = min(pieces, (t.z + 1) * perSplit);
    const uint32_t myq = lane & 31;
    const uint32_t limit = p.causal ? p.cached + min(myq, p.S - 1) : total - 1;      // last key this query sees
    const uint32_t seenByAll = p.causal ? p.cached : total - 1;                      // ... and every query

    bool seenNew = !consumer;       // the new rows' K and V are known to be there
    auto issue = [&](uint32_t h, uint32_t st) {
      const bool valid = h < end;
      if (valid && !seenNew && (h + 1) * kPieceKeys > p.cached) {
        waitRows(E + head * kHD);
        if (stage.d.in.kind != CUSYNC_POLICY_ROWSYNC) waitRows(2 * E + head * kHD);
        seenNew = true;
      }
      const uint32_t rowOff = (h * kPieceKeys + ldRow) * p.ldq;
#pragma unroll
      for (int q = 0; q < 8; q++)
        loadToLds(rLds, __builtin_amdgcn_readfirstlane(ringLds + st * kPieceBytes + q * 1024),
                  valid ? (rowOff + q * 4 * p.ldq + E + head * kHD + (((lane & 15) ^ ((4 * q + (lane >> 4)) & 15))) * 8) * 2 : kOutOfRange);
#pragma unroll
      for (int q = 0; q < 8; q++)
        loadToLds(rLds, __builtin_amdgcn_readfirstlane(ringLds + st * kPieceBytes + kPieceBytes / 2 + q * 1024),
                  valid ? (rowOff + q * 4 * p.ldq + 2 * E + head * kHD + vChunk * 8) * 2 : kOutOfRange);
    };
    issue(first, 0);
    issue(first + 4, 1);
    if (tid == 0 && round == 0) stage.finishStart(startToken, p.launched, entered);
    if (consumer) waitRows(head * kHD);
    half8 qf[8];
#pragma unroll
    for (int s = 0; s < 8; s++)
      qf[s] = __builtin_bit_cast(half8, loadChunk(rReg, myq < p.S ? ((p.cached + myq) * p.ldq + head * kHD + 16 * s + 8 * hi) * 2 : kOutOfRange));
#pragma unroll
    for (int s = 0; s < 8; s++) asm volatile("" : "+v"(qf[s]));      // waited for here, once (see attentionKernel)
    const unsigned long long tl1 = p.timeline ? wall_clock64() : 0;

    float rowMax = kMasked, rowSum = 0.0f;
    floatx16 o[4];
#pragma unroll
    for (int tt = 0; tt < 4; tt++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[tt][r] = 0.0f;

    for (uint32_t h = first, st = 0; h < end; h += 4, st ^= 1) {
      waitVmcnt<kPieceLoads>();        // this piece; the next one may still be on its way
      const char* ks = ring + st * kPieceBytes;
      const char* vs = ks + kPieceBytes / 2;
      typedef short4v __attribute__((address_space(3))) * lds_ptr;
      half8 kf[8], vf[2][4];
#pragma unroll
      for (int s = 0; s < 8; s++) kf[s] = *reinterpret_cast<const half8*>(ks + kFrag[s]);
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int tt = 0; tt < 4; tt++) {
          const char* q = vs + ((tt & 1) ? vOdd + (tt - 1) * 64 : vEven + tt * 64) + u * 16 * kRowBytes;
          const half4 l4 = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(q)));
          const half4 u4 = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(q + 8 * kRowBytes)));
          vf[u][tt] = __builtin_shufflevector(l4, u4, 0, 1, 2, 3, 4, 5, 6, 7);
        }
      floatx16 sacc[2];                // two chains of matrix instructions instead of one twice as long
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int r = 0; r < 16; r++) sacc[a][r] = 0.0f;
#pragma unroll
      for (int s = 0; s < 8; s++) sacc[s & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[s], qf[s], sacc[s & 1], 0, 0, 0);
      float sc[16];
#pragma unroll
      for (int r = 0; r < 16; r++) sc[r] = sacc[0][r] + sacc[1][r];
      if (h * kPieceKeys + kPieceKeys - 1 > seenByAll) {
        const uint32_t kv = h * kPieceKeys + 4 * hi;
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (kv + 8 * (r / 4) + (r % 4) > limit) sc[r] = kUnseen;
      }
      float pieceMax = sc[0];
#pragma unroll
      for (int r = 1; r < 16; r++) pieceMax = __builtin_fmaxf(pieceMax, sc[r]);
      pieceMax = fmaxf(pieceMax, __shfl_xor(pieceMax, 32));
      const float newMax = fmaxf(rowMax, pieceMax);
      const float alpha = __builtin_amdgcn_exp2f((rowMax - newMax) * p.scaleLog2);
      const float shift = newMax * p.scaleLog2;
      rowMax = newMax;
      half8 pf[2];
      float pieceSum = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[r], p.scaleLog2, -shift));
        pieceSum += e;
        pf[r / 8][r % 8] = (half_t)e;
      }
      rowSum = rowSum * alpha + pieceSum;
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
        for (int tt = 0; tt < 4; tt++)
#pragma unroll
          for (int r = 0; r < 16; r++) o[tt][r] *= alpha;
      }
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int tt = 0; tt < 4; tt++) o[tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[u][tt], pf[u], o[tt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);        // the piece has been read
      issue(h + 8, st);                // into the piece just read; past the end: zeros, so that every pass waits for the same count
    }
    waitVmcnt<0>();
    const unsigned long long tl2 = p.timeline ? wall_clock64() : 0;
    const AttnParams e = cusync::argumentsHere<AttnParams>(from);
    if (tid == 0) nextRaw = e.stage.drawBegin(dryXcds, noDraws);
    rowSum += __shfl_xor(rowSum, 32);

    // Four running results into one: wavefront w's [tt][g][lane] values behind one another, 16 KB each.
    __syncthreads();                   // every wavefront is out of its ring
#pragma unroll
    for (int tt = 0; tt < 4; tt++)
#pragma unroll
      for (int g = 0; g < 4; g++)
        *reinterpret_cast<floatx4*>(smem + ((wave * 16 + tt * 4 + g) * 64 + lane) * 16) =
            floatx4{o[tt][4 * g], o[tt][4 * g + 1], o[tt][4 * g + 2], o[tt][4 * g + 3]};
    sStat[0][wave][lane] = rowMax * e.scaleLog2;       // (scaled: a wavefront without keys keeps a value far below any score)
    sStat[1][wave][lane] = rowSum;
    __syncthreads();
    float m = sStat[0][0][lane], sum = 0.0f;
#pragma unroll
    for (int w = 1; w < 4; w++) m = fmaxf(m, sStat[0][w][lane]);
    floatx4 mine[4];                   // head-dim 32 * wave + 8 g + 4 hi .. + 3 of query myq
#pragma unroll
    for (int g = 0; g < 4; g++) mine[g] = floatx4{0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const float f = __builtin_amdgcn_exp2f(sStat[0][w][lane] - m);
      sum += f * sStat[1][w][lane];
#pragma unroll
      for (int g = 0; g < 4; g++) mine[g] += f * *reinterpret_cast<const floatx4*>(smem + ((w * 16 + wave * 4 + g) * 64 + lane) * 16);
    }

    bool completed = true;
    if (splits > 1) {
      // this split's share into the workspace, written through (see attentionKernel); the last to arrive adds them up
      const size_t slot = (size_t)head * e.stage.d.grid.z;
      const __amdgpu_buffer_rsrc_t rPart = makeRsrc(e.partO, e.partBytes);
      auto offO = [&](uint32_t z, int g) { return (uint32_t)(((slot + z) * (64 * kThreads) + (g * kThreads + tid) * 4) * sizeof(float)); };
      auto offS = [&](uint32_t z, int which) {
        return (uint32_t)(((char*)e.partStat - (char*)e.partO) + ((slot + z) * (2 * kThreads) + which * kThreads + lane) * sizeof(float));
      };
#pragma unroll
      for (int g = 0; g < 4; g++)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, mine[g]), rPart, (int)offO(t.z, g), 0, 16 /* sc1 */);
      if (wave == 0) {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, m), rPart, (int)offS(t.z, 0), 0, 16);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, sum), rPart, (int)offS(t.z, 1), 0, 16);
      }
      waitVmcnt<0>();
      __syncthreads();
      uint32_t* counter = e.arrivals + head;
      if (tid == 0) {
        const bool last = e.stage.countIn(counter) == splits - 1;
        if (last) { cusync::dev::storeRelaxed(counter, 0); e.stage.countSeen(); }
        sLast = last;
      }
      __syncthreads();
      completed = sLast != 0;
      if (completed) {
        constexpr uint32_t AT_ONCE = 8;
        auto loadStat = [&](uint32_t z, int which) {
          return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rPart, (int)offS(z, which), 0, 16 /* sc1 */));
        };
        // The shares are added as they arrive, eight splits at a time, the running result rescaled where a later
        // group brings a larger maximum.
        m = 2 * kMasked;
        sum = 0.0f;
#pragma unroll
        for (int g = 0; g < 4; g++) mine[g] = floatx4{0, 0, 0, 0};
        for (uint32_t z = 0; z < splits; z += AT_ONCE) {
          float zMax[AT_ONCE], zSum[AT_ONCE];
          uint4v v[AT_ONCE][4];
#pragma unroll
          for (uint32_t q = 0; q < AT_ONCE; q++) {
            const uint32_t zz = min(z + q, splits - 1);
            zMax[q] = loadStat(zz, 0);
            zSum[q] = loadStat(zz, 1);
#pragma unroll
            for (int g = 0; g < 4; g++) v[q][g] = __builtin_amdgcn_raw_buffer_load_b128(rPart, (int)offO(zz, g), 0, 16 /* sc1 */);
          }
          float newM = m;
#pragma unroll
          for (uint32_t q = 0; q < AT_ONCE; q++) newM = fmaxf(newM, zMax[q]);
          const float alpha = __builtin_amdgcn_exp2f(m - newM);
          m = newM;
          sum *= alpha;
#pragma unroll
          for (int g = 0; g < 4; g++) mine[g] *= alpha;
#pragma unroll
          for (uint32_t q = 0; q < AT_ONCE; q++) {
            const float f = z + q < splits ? __builtin_amdgcn_exp2f(zMax[q] - m) : 0.0f;
            sum += f * zSum[q];
#pragma unroll
            for (int g = 0; g < 4; g++) mine[g] += f * __builtin_bit_cast(floatx4, v[q][g]);
          }
        }
      }
    }
    if (completed && myq < e.S) {
      const float inv = 1.0f / sum;
      const __amdgpu_buffer_rsrc_t rOut = makeRsrc(e.out, e.S * e.ldo * 2);
      const uint32_t dst = (myq * e.ldo + head * kHD + 32 * wave + 4 * hi) * 2;
#pragma unroll
      for (int g = 0; g < 4; g++) {
        half4 v;
#pragma unroll
        for (int c = 0; c < 4; c++) v[c] = (half_t)(mine[g][c] * inv);
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2v, v), rOut, (int)(dst + 16 * g), 0, 16 /* sc1 */);
      }
    }
    const cusync_dim3 done = {0, head * kHD, 0};
    if (completed && e.stage.isProducer()) e.stage.post(done, 1, e.stage.storesThrough());
    else __syncthreads();
    if (tid == 0) recordTileAt(e.timeline, e.timelineCap, e.stage, e.launched, t, round, tlEntry, tl0, tl1, tl2, e.timeline ? wall_clock64() : 0);
  }
  const AttnParams atEnd = cusync::argumentsHere<AttnParams>(from);
  atEnd.stage.leave(atEnd.launched);
}

}  // namespace attn
}  // namespace cusync
