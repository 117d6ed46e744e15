// gemm_wr (gemm_wr.h) for fp16 activations.
#include "gemm_wr_launch.h"

namespace ofq {
int launch_gemm_wr_f16(hipStream_t st, const LinearArgs& a, const WrPlan& plan, float* partials) {
  return launch_wr_t<f16, MfmaF16>(st, a, plan, partials);
}
}  // namespace ofq
