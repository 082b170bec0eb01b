// Launch of the GEMM that holds its weights in registers (gemm_resident_kernel.h).
#include "gemm_resident_kernel.h"
#include "gemm_resident.h"
#include "rt_internal.h"

namespace cusync {
namespace gemm {

template<class C>
static bool ready() {
  return !CUSYNC_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gemmResidentKernel<C>), hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES));
}
bool residentReady(uint32_t columns) { return columns == 64 ? ready<ResidentCfg<64>>() : ready<ResidentCfg<128>>(); }

template<class C>
static cusync_error launchResident(const cusync_gemm_args* a, void* stream) {
  const cusync_stage_desc& s = a->stage;
  const bool waits = s.in.kind != CUSYNC_POLICY_NOSYNC;
  if (a->M == 0 || a->M > C::MAX_ROWS || a->K > C::MAX_K || a->split_k != 1 || a->epilogue != CUSYNC_EPILOGUE_NONE || a->a_mode != CUSYNC_A_PLAIN ||
      s.out.kind != CUSYNC_POLICY_NOSYNC ||
      (waits && ((s.in.kind != CUSYNC_POLICY_ROWSYNC && s.in.kind != CUSYNC_POLICY_TILESYNC) || !(s.opts & CUSYNC_OPT_REORDER_TILE_LOADS)))) {
    rt::setError("gemm: not a problem for weights held in registers");
    return CUSYNC_ERROR_NOT_INITIALIZED;
  }
  GemmParams p = {};
  p.stage.d = s;
  p.stage.lineAligned = waits && !rt::forceAcquire() && (uintptr_t)a->A % 128 == 0 && (a->lda * 2) % 128 == 0 &&
                        (s.in.kind == CUSYNC_POLICY_ROWSYNC || (s.in.tileN * 2) % 128 == 0);
  p.stage.releaseAll = rt::forceRelease();
  p.launched = residentGrid(a->N, C::BN).x;
  p.stage.prepare(p.launched);
  p.M = a->M; p.N = a->N; p.K = a->K;
  p.A = (const half_t*)a->A; p.lda = a->lda;
  p.B = (const half_t*)a->B; p.ldb = a->ldb;
  p.D = (half_t*)a->D; p.ldd = a->ldd;
  p.kPerSlice = (a->K + C::WAVES * C::KS - 1) / (C::WAVES * C::KS) * C::KS;       // columns of K to a wavefront
  rt::timeline(&p.timeline, &p.timelineCap);
  hipLaunchKernelGGL((gemmResidentKernel<C>), dim3(p.launched), dim3(C::THREADS), C::LDS_BYTES, (hipStream_t)stream, p);
  return CUSYNC_HIP(hipGetLastError()) ? CUSYNC_ERROR_DEVICE : CUSYNC_SUCCESS;
}

cusync_error residentRun(const cusync_gemm_args* a, uint32_t columns, void* stream) {
  return columns == 64 ? launchResident<ResidentCfg<64>>(a, stream) : launchResident<ResidentCfg<128>>(a, stream);
}

}  // namespace gemm
}  // namespace cusync
