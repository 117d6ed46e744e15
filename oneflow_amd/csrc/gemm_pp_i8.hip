// gemm_pp (gemm_pp.h) on int8 operands, with matmul_quant's epilogue.
#include "gemm_pp.h"
#include "ofq_internal.h"

namespace ofq {
namespace {
template<typename T>
int launch(hipStream_t st, const void* a, const void* b, const float* a_scale, const float* b_scale,
           const void* bias, void* out, int64_t m, int64_t n, int64_t k, int width) {
  typedef typename TT<T>::storage S;
  typename EpScale<T>::Params ep{a_scale, b_scale, static_cast<const S*>(bias), static_cast<S*>(out)};
  return launch_pp<MfmaI8, EpScale<T>>(st, a, b, k, ep, m, n, width);
}
}  // namespace

int launch_gemm_pp_i8(hipStream_t st, const void* a, const void* b, const float* a_scale,
                      const float* b_scale, const void* bias, void* out, int out_dtype, int64_t m,
                      int64_t n, int64_t k, int width) {
  switch (out_dtype) {
    case OFQ_F16: return launch<f16>(st, a, b, a_scale, b_scale, bias, out, m, n, k, width);
    case OFQ_BF16: return launch<bf16>(st, a, b, a_scale, b_scale, bias, out, m, n, k, width);
    default: return launch<float>(st, a, b, a_scale, b_scale, bias, out, m, n, k, width);
  }
}
}  // namespace ofq
