// Kernel instantiations and launchers of the GEMM in arithmetic F32 (FP32 MFMA).
#include "gemm_direct.h"

namespace tnx {

void gemm_direct_f32(const GemmDesc& d, const GemmArgs& g, hipStream_t s) {
  if (d.ta == DT::F64 && d.tb == DT::F64) return gemm_direct_run<1, double, double>(d, g, s);
  if (d.ta == DT::F64) return gemm_direct_run<1, double, float>(d, g, s);
  if (d.tb == DT::F64) return gemm_direct_run<1, float, double>(d, g, s);
  return gemm_direct_run<1, float, float>(d, g, s);
}

void gemm_launch_f32(const GemmDesc& d, const GemmArgs& g, int splits, hipStream_t s) {
  gemm_launch_index<1, void, void>(0, d, g, splits, s);
}

}  // namespace tnx
