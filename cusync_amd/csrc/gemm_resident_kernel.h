// A GEMM of few rows whose weights fit the register files: each workgroup holds its columns of B, all of K, before A is there.
//
// For the last stage of a chain.  The tiled kernels (DmaCfg::AHEAD) have three stages of their ring, a quarter of a slice's
// weights, under way when the producer posts; the rest streams behind the wait, and the k-slices that streaming needs come
// together through memory.  The output projection of 12 heads is 37.7 MB, 196 KB for each of 192 workgroups: a wavefront takes an
// eighth of K, at most 192 rows of 64 columns, into 96 registers (of 128 columns: 192), and turns them into MFMA operands in place.
// What is left behind the wait is A (16 rows at a time, straight into LDS in the order the fragments are read, the next 16 while
// these are multiplied), 24 or 48 MFMAs a wavefront, the sum over the eight wavefronts through LDS, and the store: a chain of round
// trips, 3 us for up to 16 rows, 1.7 us for each further 16, which bounds it.  K goes to the wavefronts the same way whatever the
// columns, so results do not depend on them.
//
// The layer, 12 heads, hidden 12288, us, tiles in k-slices -> this, each pass on other operands than the one before: behind 2000 rows
// under RowSync 1 row 59.0 -> 52.3, 16 60.3 -> 54.4, 32 61.9 -> 57.6, 64 77.7 -> 73.4, 112 93.8 -> 92.5; TileSync 16 rows 58.2 -> 52.2; without a
// cache under RowSync 16 rows 53.7 -> 51.0, 64 65.0 -> 60.9, 96 82.1 -> 76.8; in stream order, where nothing is read ahead and the gain is the k-slices'
// exchange, 1 row 56.6 -> 53.1, 16 57.3 -> 54.9, 32 58.7 -> 57.7, 64 69.4 -> 66.0, 112 85.2 -> 85.1.  (Which projections: weightsFitRegisters.)
//
// A workgroup has a CU's LDS to itself although it would do with half: two to a CU, half the CUs read all the weights, and 16 rows
// behind 2048 took 61.4 us.
#pragma once

#include "gemm_kernel_dma.h"

namespace cusync {
namespace gemm {

// BN: columns of a workgroup, 64 or 128.
template<int BN_>
struct ResidentCfg {
  static constexpr int BN = BN_, COLS = BN / 16, ROWS = 16, WAVES = 8, THREADS = WAVES * 64, KS = 32, STEPS = 6;
  static constexpr uint32_t MAX_ROWS = 112, MAX_K = WAVES * STEPS * KS;
  static constexpr int A_BYTES = STEPS * 1024;                    // of a wavefront: 16 rows of its k, a KiB per k-step
  static constexpr int BUFFERS = 2;                               // 16 rows being multiplied, 16 on their way
  static constexpr int PITCH = BN + 4;                            // floats
  static constexpr int PARTS = WAVES / 2, PART_FLOATS = ROWS * PITCH;
  static constexpr int STORING = ROWS * BN / 4 / 64;              // wavefronts that store, one store for 16 rows
  static constexpr int LDS_BYTES = BUFFERS * WAVES * A_BYTES + PARTS * PART_FLOATS * 4;
};

template<class C>
__global__ __launch_bounds__(C::THREADS, 2) void gemmResidentKernel(GemmParams p) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  float* parts = reinterpret_cast<float*>(smem + C::BUFFERS * C::WAVES * C::A_BYTES);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t slot = lane & 15, group = lane >> 4;
  const cusync::DynStage& stage = p.stage;
  const bool consumer = stage.isConsumer();
  const unsigned long long tlEntry = p.timeline ? wall_clock64() : 0;
  const uint32_t n0 = blockIdx.x * C::BN;

  // k-step t of a wavefront: 32 rows of B from kFirst + 32 t on, eight of them to each of the four lane groups; whole groups
  // are inside K or not.
  const uint32_t kWave = p.kPerSlice, kFirst = wave * kWave;
  const int steps = kFirst < p.K ? (int)((min(kWave, p.K - kFirst) + C::KS - 1) / C::KS) : 0;

  // Lane `slot` of a group takes COLS columns next to one another of the group's eight rows: a row is BN columns of the 16 lanes.
  typedef std::conditional_t<C::COLS == 8, uint4v, uint2v> Piece;
  Piece w[C::STEPS][8];
  const __amdgpu_buffer_rsrc_t rB = makeRsrc(p.B, p.K * p.ldb * 2);
  auto loadWeights = [&] {
#pragma unroll
    for (int t = 0; t < C::STEPS; t++) {
      const uint32_t k = kFirst + t * C::KS + group * 8;
      const uint32_t off = t < steps && k < p.K && n0 + C::COLS * slot < p.N ? (k * p.ldb + n0 + C::COLS * slot) * 2 : kOutOfRange;
#pragma unroll
      for (int j = 0; j < 8; j++)
        if constexpr (C::COLS == 8) w[t][j] = __builtin_amdgcn_raw_buffer_load_b128(rB, (int)off, (int)(j * p.ldb * 2), 2 /* nt: read once */);
        else w[t][j] = __builtin_bit_cast(uint2v, __builtin_amdgcn_raw_buffer_load_b64(rB, (int)off, (int)(j * p.ldb * 2), 2));
    }
  };
  // Fragment c of a step: element j is row j, column COLS slot + c.  A column of the MFMA's operand is any column of B, so
  // column tile c takes the columns that are c modulo COLS, and nothing moves between lanes.
  auto fragment = [&](int t, int c) {
    uint4v f;
#pragma unroll
    for (int r = 0; r < 4; r++)
      f[r] = __builtin_amdgcn_perm(w[t][2 * r + 1][c / 2], w[t][2 * r][c / 2], c & 1 ? 0x07060302u : 0x05040100u);
    return f;
  };
  uint4v frag[C::STEPS][C::COLS];
  auto turn = [&] {
#pragma unroll
    for (int t = 0; t < C::STEPS; t++) {
#pragma unroll
      for (int c = 0; c < C::COLS; c++) frag[t][c] = fragment(t, c);
#pragma unroll
      for (int c = 0; c < C::COLS; c++) asm volatile("" : "+v"(frag[t][c]));
    }
  };

  const uint4v rA = rawRsrc(p.A, p.M * p.lda * 2);
  const uint32_t aBase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * C::A_BYTES;
  // (The thread's index is made opaque where it is used, so that nothing is worked out of it ahead: there are no registers to
  // keep that in beside the weights.)
  auto loadA = [&](uint32_t m0) {
    int l = lane;
    asm volatile("" : "+v"(l));
    const uint32_t k = kFirst + (l >> 4) * 8, row = m0 + (l & 15), to = aBase + (m0 / C::ROWS % C::BUFFERS) * (C::WAVES * C::A_BYTES);
#pragma unroll
    for (int t = 0; t < C::STEPS; t++)
      if (t < steps)
        loadToLds(rA, __builtin_amdgcn_readfirstlane(to + t * 1024), row < p.M && k + t * C::KS < p.K ? (row * p.lda + k + t * C::KS) * 2 : kOutOfRange);
  };

  // (A consumer comes here with ReorderTileLoads only: the weights are not its producer's stream's to write.)
  if (!consumer) loadA(0);
  loadWeights();
  turn();
  if (consumer) {
    if (wave == 0) {
      const uint32_t tmq = stage.d.in.tileM, tnq = stage.d.in.tileN;
      if (stage.d.in.kind == CUSYNC_POLICY_ROWSYNC) {
        stage.waitWaveRows(0, p.M - 1, tmq, 0, 1);
      } else {
        const uint32_t cols = (p.K + tnq - 1) / tnq;
        for (uint32_t col = 0; col < cols;) col += stage.waitWaveAheadRows(0, p.M - 1, tmq, col * tnq, tnq, cols - col);
      }
    }
    __syncthreads();
    loadA(0);
  }
  const unsigned long long tl1 = p.timeline ? wall_clock64() : 0;

  const __amdgpu_buffer_rsrc_t rD = makeRsrc(p.D, p.M * p.ldd * 2);
  for (uint32_t m0 = 0; m0 < p.M; m0 += C::ROWS) {
    if (m0 == 0) waitVmcnt<0>();
    else if (wave < C::STORING) waitVmcnt<1>();      // the store of the rows before is behind these rows' loads
    else waitVmcnt<0>();
    if (m0 + C::ROWS < p.M) loadA(m0 + C::ROWS);
    int id = tid;
    asm volatile("" : "+v"(id));
    floatx4 acc[C::COLS];
#pragma unroll
    for (int c = 0; c < C::COLS; c++) acc[c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const char* rows = smem + (m0 / C::ROWS % C::BUFFERS) * (C::WAVES * C::A_BYTES) + wave * C::A_BYTES + (id & 63) * 16;
#pragma unroll
    for (int t = 0; t < C::STEPS; t++) {
      if (t >= steps) continue;
      const half8 a = *reinterpret_cast<const half8*>(rows + t * 1024);
#pragma unroll
      for (int c = 0; c < C::COLS; c++) acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, frag[t][c]), a, acc[c], 0, 0, 0);
    }
    // Register r of column tile c: row `slot` of A, column COLS (4 group + r) + c.  Wavefronts 4 to 7 hand their sums to 0 to 3,
    // which add them to theirs; the four are added up by wavefront, four columns a thread.
    float* mine = parts + (wave % C::PARTS) * C::PART_FLOATS + (id & 15) * C::PITCH + 4 * C::COLS * ((id >> 4) & 3);
    if (wave >= C::PARTS) {
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int h = 0; h < C::COLS; h += 4) *reinterpret_cast<floatx4*>(mine + C::COLS * r + h) = floatx4{acc[h][r], acc[h + 1][r], acc[h + 2][r], acc[h + 3][r]};
    }
    __syncthreads();
    if (wave < C::PARTS) {
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int h = 0; h < C::COLS; h += 4) {
          floatx4 v = *reinterpret_cast<const floatx4*>(mine + C::COLS * r + h);
#pragma unroll
          for (int c = 0; c < 4; c++) v[c] += acc[h + c][r];
          *reinterpret_cast<floatx4*>(mine + C::COLS * r + h) = v;
        }
    }
    __syncthreads();
    if (wave < C::STORING) {
      const uint32_t row = id / (C::BN / 4), col = id % (C::BN / 4) * 4;
      floatx4 sum = *reinterpret_cast<const floatx4*>(parts + row * C::PITCH + col);
#pragma unroll
      for (int q = 1; q < C::PARTS; q++) {
        const floatx4 v = *reinterpret_cast<const floatx4*>(parts + q * C::PART_FLOATS + row * C::PITCH + col);
#pragma unroll
        for (int c = 0; c < 4; c++) sum[c] += v[c];
      }
      half4 o;
#pragma unroll
      for (int c = 0; c < 4; c++) o[c] = (half_t)sum[c];
      const int off = m0 + row < p.M && n0 + col < p.N ? (int)(((m0 + row) * p.ldd + n0 + col) * 2) : (int)kOutOfRange;
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2v, o), rD, off, 0, 16 /* sc1: the stage stamps its end */);
    }
    if (m0 + C::ROWS < p.M) __syncthreads();
  }
  if (tid == 0 && p.timeline) {
    const unsigned long long tl2 = wall_clock64();
    recordTile(p, cusync_dim3{blockIdx.x, 0, 0}, 0, tlEntry, tlEntry, tl1, tl2, tl2);
  }
  stage.leave(p.launched);
}

}  // namespace gemm
}  // namespace cusync
