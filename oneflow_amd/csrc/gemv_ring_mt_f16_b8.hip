// gemv_ring_mt (gemv_ring_mt.h) for fp16 activations and 8-bit codes.
#include "gemv_ring_mt_launch.h"

namespace ofq {

int launch_gemv_ring_mt_f16_b8(hipStream_t st, const LinearJob& job, const RingMtPlan& plan) {
  return launch_ring_mt_t<f16, 8>(st, job, plan);
}

}  // namespace ofq
