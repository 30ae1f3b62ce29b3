// Kernel instantiations and launchers of the GEMM in arithmetic F64 (FP64 MFMA).
#include "gemm_direct.h"

namespace tnx {

void gemm_direct_f64(const GemmDesc& d, const GemmArgs& g, hipStream_t s) {
  // (F64, F64) and (F64, F32): the pairs gemm_direct_ok admits for F64
  if (d.tb == DT::F64) return gemm_direct_run<0, double, double>(d, g, s);
  return gemm_direct_run<0, double, float>(d, g, s);
}

void gemm_launch_f64(const GemmDesc& d, const GemmArgs& g, int splits, hipStream_t s) {
  gemm_launch_index<0, void, void>(0, d, g, splits, s);
}

}  // namespace tnx
