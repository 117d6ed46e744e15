// gemv_flow (gemv_flow.h) for bf16 activations and 8-bit codes.
#include "gemv_flow_launch.h"

namespace ofq {

int launch_gemv_flow_bf16_b8(hipStream_t st, const LinearJob& job, const FlowPlan& plan) {
  return launch_flow_t<bf16, 8>(st, job, plan);
}

}  // namespace ofq
