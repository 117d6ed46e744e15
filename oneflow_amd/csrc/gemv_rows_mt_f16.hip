// gemv_rows_mt (gemv_rows.h) for fp16 activations.
#include "gemv_rows_mt_launch.h"

namespace ofq {

int launch_gemv_mt_f16(hipStream_t st, const LinearJob& job, const RowsMtPlan& plan) {
  return launch_rows_mt_plan<f16>(st, job, plan);
}

}  // namespace ofq
