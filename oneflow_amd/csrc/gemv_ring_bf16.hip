// gemv_ring (gemv_ring.h) for bf16 activations.
#include "gemv_ring_launch.h"

namespace ofq {

int launch_gemv_ring_bf16(hipStream_t st, const LinearJob& job, const RingPlan& plan) {
  return launch_ring_t<bf16>(st, job, plan);
}

}  // namespace ofq
