// gemm_wr (gemm_wr.h) for bf16 activations.
#include "gemm_wr_launch.h"

namespace ofq {
int launch_gemm_wr_bf16(hipStream_t st, const LinearArgs& a, const WrPlan& plan, float* partials) {
  return launch_wr_t<bf16, MfmaBF16>(st, a, plan, partials);
}
}  // namespace ofq
