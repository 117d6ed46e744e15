// gemv_rows_mt (gemv_rows.h) for bf16 activations.
#include "gemv_rows_mt_launch.h"

namespace ofq {

int launch_gemv_mt_bf16(hipStream_t st, const LinearJob& job, const RowsMtPlan& plan) {
  return launch_rows_mt_plan<bf16>(st, job, plan);
}

}  // namespace ofq
