// gemv_ring_mt (gemv_ring_mt.h) for bf16 activations and 4-bit codes.
#include "gemv_ring_mt_launch.h"

namespace ofq {

int launch_gemv_ring_mt_bf16_b4(hipStream_t st, const LinearJob& job, const RingMtPlan& plan) {
  return launch_ring_mt_t<bf16, 4>(st, job, plan);
}

}  // namespace ofq
