// Polybench group: constructors and setUp/updateChecksum/tearDown follow
// src/polybench/POLYBENCH_GEMM.cpp:22-96 and POLYBENCH_JACOBI_2D.cpp:22-95.
#include "polybench/Polybench.hpp"

#include <cmath>
#include <vector>

#include "Autotune.hpp"

#include "stream/Stream.hpp"

namespace rajaperf {
namespace polybench {

// ---- GEMM ------------------------------------------------------------------------
POLYBENCH_GEMM::POLYBENCH_GEMM(const RunParams& params) : KernelBase(Polybench_GEMM, params) {
  const Index_type ni_default = 1000, nj_default = 1000, nk_default = 1200;
  setDefaultProblemSize(ni_default * nj_default);
  setDefaultReps(4);
  m_ni = static_cast<Index_type>(std::sqrt(double(getTargetProblemSize())) + std::sqrt(2.0) - 1);
  m_nj = m_ni;
  m_nk = params.getNk() > 0 ? params.getNk() : Index_type(double(nk_default) / ni_default * m_ni);
  // Suite constants (POLYBENCH_GEMM.cpp:35-36); the seeded workload uses 1.5 / 1.2;
  // --alpha / --beta override either.
  m_alpha = params.getInputMode() == RunParams::SeededInputs ? 1.5 : 0.62;
  m_beta = params.getInputMode() == RunParams::SeededInputs ? 1.2 : 1.002;
  if (params.hasGemmAlpha()) m_alpha = params.getGemmAlpha();
  if (params.hasGemmBeta()) m_beta = params.getGemmBeta();
  setActualProblemSize(m_ni * m_nj);
  setItsPerRep(m_ni * m_nj);
  setKernelsPerRep(1);
  setBytesReadPerRep(1 * sizeof(Real_type) * m_ni * m_nk + 1 * sizeof(Real_type) * m_nj * m_nk);
  setBytesWrittenPerRep(1 * sizeof(Real_type) * m_ni * m_nj);
  setBytesAtomicModifyWrittenPerRep(0);
  setFLOPsPerRep((1 + 3 * m_nk) * m_ni * m_nj);
  checksum_scale_factor = 0.001 * (static_cast<Checksum_type>(getDefaultProblemSize()) / getActualProblemSize());
  setComplexity(Complexity::N_to_the_three_halves);
  setVariantDefined(MI355X_Native);
}
void POLYBENCH_GEMM::setMI355XTuningDefinitions(VariantID vid) {
  addVariantTuningName(vid, "default");  // FP64 on the MFMA f64 units
  addVariantTuningName(vid, "naive");    // one thread per C element, the plain FP64 comparator
  addVariantTuningName(vid, "mixed");    // int8 MFMA, one GEMM per modulus (13 at nk = 4096), FP64 result
}
void POLYBENCH_GEMM::setUp(VariantID, size_t) {
  allocAndInitData(m_A, Size_type(m_ni * m_nk), -1.0, 1.0);
  allocAndInitData(m_B, Size_type(m_nk * m_nj), -1.0, 1.0);
  allocAndInitDataConst(m_C, Size_type(m_ni * m_nj), 0.0);
}
void POLYBENCH_GEMM::updateChecksum(VariantID vid, size_t t) {
  checksum[vid][t] += calcChecksum(m_C, Size_type(m_ni * m_nj), Real_type(checksum_scale_factor));
}
void POLYBENCH_GEMM::tearDown(VariantID, size_t) {
  deallocData(m_A);
  deallocData(m_B);
  deallocData(m_C);
}
void POLYBENCH_GEMM::runMI355XVariant(VariantID, size_t tune_idx) {
  const Index_type reps = getRunReps();
  if (tune_idx == 2) {  // the residues. scratch is allocated outside the timed reps
    const size_t bytes = rpx_gemm_mixed_scratch_bytes(m_ni, m_nj, m_nk, 0);
    char* scratch = nullptr;
    allocData(scratch, Size_type(bytes));
    timedReps(reps, [&](RepIndex_type) {
      rpxCheck(rpx_gemm_mixed_f64(m_C, m_A, m_B, m_alpha, m_beta, m_ni, m_nj, m_nk, 0, scratch, bytes, stream()),
               "GEMM mixed");
    });
    deallocData(scratch);
    return;
  }
  rpx_tuning tune = defaultTuning();
  if (tune_idx == 1) tune.flags |= RPX_TUNE_NAIVE;
  timedReps(reps, [&](RepIndex_type) {
    rpxCheck(rpx_gemm_f64(m_C, m_A, m_B, m_alpha, m_beta, m_ni, m_nj, m_nk, &tune, stream()), "GEMM");
  });
}

// ---- JACOBI_2D -------------------------------------------------------------------
POLYBENCH_JACOBI_2D::POLYBENCH_JACOBI_2D(const RunParams& params) : KernelBase(Polybench_JACOBI_2D, params) {
  const Index_type N_default = 1002;
  setDefaultProblemSize((N_default - 2) * (N_default - 2));
  setDefaultReps(50);
  m_N = static_cast<Index_type>(std::sqrt(double(getTargetProblemSize())) + 2 + std::sqrt(2.0) - 1);
  m_tsteps = params.getTsteps() > 0 ? params.getTsteps() : 40;
  setActualProblemSize((m_N - 2) * (m_N - 2));
  setItsPerRep(m_tsteps * (2 * (m_N - 2) * (m_N - 2)));
  setKernelsPerRep(2);
  setBytesReadPerRep((1 * sizeof(Real_type) * (m_N * m_N - 4) + 1 * sizeof(Real_type) * (m_N * m_N - 4)) *
                     m_tsteps);
  setBytesWrittenPerRep(
      (1 * sizeof(Real_type) * (m_N - 2) * (m_N - 2) + 1 * sizeof(Real_type) * (m_N - 2) * (m_N - 2)) * m_tsteps);
  setBytesAtomicModifyWrittenPerRep(0);
  setFLOPsPerRep(m_tsteps * (5 * (m_N - 2) * (m_N - 2) + 5 * (m_N - 2) * (m_N - 2)));
  checksum_scale_factor = 0.0001 * (static_cast<Checksum_type>(getDefaultProblemSize()) / getActualProblemSize());
  setComplexity(Complexity::N);
  setVariantDefined(MI355X_Native);
}
void POLYBENCH_JACOBI_2D::setMI355XTuningDefinitions(VariantID vid) {
  addVariantTuningName(vid, "default");    // tile or chunk, and time steps per fused launch, by N and tsteps
  addVariantTuningName(vid, "depth_2");    // two time steps per fused launch
  addVariantTuningName(vid, "depth_1");    // one time step per fused launch
  addVariantTuningName(vid, "two_sweep");  // one launch per sweep, as the suite's kernels
  addVariantTuningName(vid, "two_sweep_rows_32");
  addVariantTuningName(vid, "auto");       // the default and fused depth x tile rows, measured
}
void POLYBENCH_JACOBI_2D::setUp(VariantID, size_t) {
  const Size_type nn = Size_type(m_N * m_N);
  allocData(m_Ainit, nn);
  allocData(m_Binit, nn);
  if (seededInputs()) {  // interior uniform [0,1), zero boundary
    detail::initDataSeededGridDevice(m_Ainit, m_N, run_params.getSeed());
    detail::initDataSeededGridDevice(m_Binit, m_N, run_params.getSeed());
  } else {
    detail::initDataDevice(m_Ainit, nn);
    detail::initDataDevice(m_Binit, nn);
  }
  allocData(m_A, nn);
  allocData(m_B, nn);
}
void POLYBENCH_JACOBI_2D::updateChecksum(VariantID vid, size_t t) {
  checksum[vid][t] += calcChecksum(m_A, Size_type(m_N * m_N), Real_type(checksum_scale_factor));
  checksum[vid][t] += calcChecksum(m_B, Size_type(m_N * m_N), Real_type(checksum_scale_factor));
}
void POLYBENCH_JACOBI_2D::tearDown(VariantID, size_t) {
  deallocData(m_A);
  deallocData(m_B);
  deallocData(m_Ainit);
  deallocData(m_Binit);
}
void POLYBENCH_JACOBI_2D::runMI355XVariant(VariantID, size_t tune_idx) {
  const Index_type reps = getRunReps();
  rpx_tuning tune = defaultTuning();
  const bool fused = tune_idx <= 2;
  if (tune_idx == 1) tune.depth = 2;
  if (tune_idx == 2) tune.depth = 1;
  if (tune_idx == 4) tune.items_per_thread = 32;
  // POLYBENCH_JACOBI_2D_DATA_SETUP copies the initial grids before the timer.
  const Size_type bytes = Size_type(m_N * m_N) * sizeof(Real_type);
  rpxCheck(rpx_memcpy_d2d(m_A, m_Ainit, bytes, nullptr), "JACOBI_2D copy");
  rpxCheck(rpx_memcpy_d2d(m_B, m_Binit, bytes, nullptr), "JACOBI_2D copy");
  const size_t sb = (fused || tune_idx == 5) ? rpx_jacobi2d_fused_scratch_bytes(m_N) : 0;
  void* scratch = sb ? detail::deviceAlloc(sb) : nullptr;
  if (tune_idx == 5) {
    // Trials advance copies of the initial grids, so A and B still start
    // from DATA_SETUP's values when the timed reps begin.
    std::vector<TuneCandidate> cands{{"default", defaultTuning()}};
    for (int depth = 1; depth <= 4; ++depth)
      for (int rows : {8, 16, 54, 99, 144}) {
        if (depth == 4 && rows < 54) continue;  // depth 4 runs streaming chunks only
        rpx_tuning t = defaultTuning();
        t.depth = depth;
        t.items_per_thread = rows;
        cands.push_back({"depth_" + std::to_string(depth) + "_rows_" + std::to_string(rows), t});
      }
    auto tA = static_cast<Real_ptr>(detail::deviceAlloc(bytes));
    auto tB = static_cast<Real_ptr>(detail::deviceAlloc(bytes));
    rpxCheck(rpx_memcpy_d2d(tA, m_A, bytes, nullptr), "JACOBI_2D copy");
    rpxCheck(rpx_memcpy_d2d(tB, m_B, bytes, nullptr), "JACOBI_2D copy");
    tune = Autotuner::instance()
               .choose(getName(), "N=" + std::to_string(m_N) + ",tsteps=" + std::to_string(m_tsteps), cands,
                       [&](const rpx_tuning& t) {
                         rpxCheck(rpx_jacobi2d_fused_f64(tA, tB, m_N, m_tsteps, scratch, sb, &t, nullptr),
                                  "JACOBI_2D");
                       })
               .tuning;
    detail::deviceFree(tA);
    detail::deviceFree(tB);
  }
  const bool run_fused = fused || tune_idx == 5;
  timedReps(reps, [&](RepIndex_type) {
    if (run_fused)
      rpxCheck(rpx_jacobi2d_fused_f64(m_A, m_B, m_N, m_tsteps, scratch, sb, &tune, stream()), "JACOBI_2D");
    else rpxCheck(rpx_jacobi2d_f64(m_A, m_B, m_N, m_tsteps, &tune, stream()), "JACOBI_2D");
  });
  if (scratch) detail::deviceFree(scratch);
}

}  // namespace polybench
}  // namespace rajaperf
