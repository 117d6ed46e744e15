// gemm_pp (gemm_pp.h) on bf16 operands.
#include "gemm_pp.h"
#include "ofq_internal.h"

namespace ofq {
int launch_gemm_pp_bf16(hipStream_t st, const void* x, const void* w, const void* bias, void* out,
                    int64_t m, int64_t n, int64_t k, int width) {
  typedef TT<bf16>::storage S;
  EpBias<bf16>::Params ep{static_cast<const S*>(bias), static_cast<S*>(out)};
  return launch_pp<MfmaBF16, EpBias<bf16>>(st, x, w, k * 2, ep, m, n, width);
}
}  // namespace ofq
