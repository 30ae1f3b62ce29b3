// Kernel instantiations and launchers of the GEMM in arithmetic F64 (FP64 MFMA).
#include "gemm_direct.h"

namespace tnx {

void gemm_direct_f64(const GemmDesc& d, const GemmArgs& g, hipStream_t s) {
  if (d.ta == DT::F64 && d.tb == DT::F64) return gemm_direct_run<0, double, double>(d, g, s);
  if (d.ta == DT::F64) return gemm_direct_run<0, double, float>(d, g, s);
  if (d.tb == DT::F64) return gemm_direct_run<0, float, double>(d, g, s);
  return gemm_direct_run<0, float, float>(d, g, s);
}

void gemm_launch_f64(const GemmDesc& d, const GemmArgs& g, int splits, hipStream_t s) {
  gemm_launch_index<0, void, void>(0, d, g, splits, s);
}

}  // namespace tnx
