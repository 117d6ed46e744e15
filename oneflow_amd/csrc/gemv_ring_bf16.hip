#include "gemv_ring_launch.h"

namespace ofq {

int launch_gemv_ring_bf16(hipStream_t st, const LinearArgs* pr, int count, bool glu, void* y, int act) {
  return launch_ring_t<bf16>(st, pr, count, glu, y, act);
}

}  // namespace ofq
