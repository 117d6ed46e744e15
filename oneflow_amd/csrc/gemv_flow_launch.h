// Launch of gemv_flow (gemv_flow.h) for one T and width; included by one source file for each so that they compile
// side by side.
#pragma once

#include "gemv_flow.h"
#include "ofq_internal.h"

namespace ofq {
namespace {

template<typename T, int BITS, bool SIGNED, int ZMODE, bool LATE, int MX, int TL, int NW>
int launch_flow_inst(hipStream_t st, const LinearJob& job, const FlowPlan& plan) {
  const LinearArgs& a = job.pr[0];
  FlowArgs p{};
  p.M = (int)a.m;
  p.K = (int)a.k;
  p.group_size = (int)a.group_size;
  p.gs_shift = -1;
  for (int s = 0; s < 31; ++s)
    if (((int64_t)1 << s) == a.group_size) p.gs_shift = s;
  p.rows_per_block = plan.rows_per_block;
  const uint16_t* x = static_cast<const uint16_t*>(a.x);
  static std::atomic<uint64_t> allowed{0}, allowed_grouped{0}, allowed_glu{0};  // devices: LDS limit raised
  if (job.glu) {
    if constexpr (TL <= 3) {
      auto kern = gemv_flow_glu<T, BITS, SIGNED, ZMODE, LATE, MX, TL, NW>;
      if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed_glu)) return OFQ_ERR_LAUNCH;
      kern<<<plan.grid, NW * 64, plan.lds, st>>>(x, rows_mat(a), rows_mat(job.pr[1]), (int)a.n,
                                                 static_cast<uint16_t*>(job.y), job.act, p);
    } else {
      return OFQ_ERR_UNSUPPORTED;
    }
  } else if (job.count > 1) {
    auto kern = gemv_flow_grouped<T, BITS, SIGNED, ZMODE, LATE, MX, TL, NW>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed_grouped)) return OFQ_ERR_LAUNCH;
    GemvGroup g{};
    fill_group(g, job.pr, job.count, plan.rows_per_block);
    kern<<<plan.grid, NW * 64, plan.lds, st>>>(g, p);
  } else {
    // (a tile-major copy has groups of whole chunks and up to 64 rows a block)
    if constexpr (BITS == 4 && TT<T>::dtype == OFQ_F16 && MX <= 2 && TL <= 4 && (LATE || ZMODE != kZeroNone)) {
      if (plan.tiled) {
        auto kern = gemv_flow<T, BITS, SIGNED, ZMODE, LATE, true, MX, TL, NW>;
        static std::atomic<uint64_t> allowed_tiled{0};
        if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed_tiled)) return OFQ_ERR_LAUNCH;
        kern<<<plan.grid, NW * 64, plan.lds, st>>>(x, rows_mat(a), (int)a.n, p);
        return ofq_check_launch();
      }
    }
    if (plan.tiled) return OFQ_ERR_UNSUPPORTED;
    auto kern = gemv_flow<T, BITS, SIGNED, ZMODE, LATE, false, MX, TL, NW>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed)) return OFQ_ERR_LAUNCH;
    kern<<<plan.grid, NW * 64, plan.lds, st>>>(x, rows_mat(a), (int)a.n, p);
  }
  return ofq_check_launch();
}

template<typename T, int BITS, bool SIGNED, int ZMODE, bool LATE = false>
int launch_flow_variant(hipStream_t st, const LinearJob& job, const FlowPlan& plan) {
#define OFQ_L(MXV, TLV, NWV) \
  if (plan.mx == MXV && plan.tl == TLV && plan.nw == NWV) \
    return launch_flow_inst<T, BITS, SIGNED, ZMODE, LATE, MXV, TLV, NWV>(st, job, plan);
  OFQ_L(1, 1, 8) OFQ_L(1, 2, 8) OFQ_L(1, 3, 8) OFQ_L(1, 4, 8) OFQ_L(1, 5, 8) OFQ_L(1, 6, 8)
  OFQ_L(2, 1, 8) OFQ_L(2, 2, 8) OFQ_L(2, 3, 8) OFQ_L(2, 4, 8) OFQ_L(2, 5, 8)
  OFQ_L(1, 1, 6) OFQ_L(1, 2, 6) OFQ_L(1, 3, 6) OFQ_L(1, 4, 6) OFQ_L(1, 5, 6) OFQ_L(1, 6, 6)
  OFQ_L(2, 1, 6) OFQ_L(2, 2, 6) OFQ_L(2, 3, 6) OFQ_L(2, 4, 6) OFQ_L(2, 5, 6)
  if constexpr (!LATE) {
    OFQ_L(4, 1, 8) OFQ_L(4, 2, 8) OFQ_L(4, 3, 8) OFQ_L(4, 4, 8)
    OFQ_L(6, 1, 8) OFQ_L(6, 2, 8) OFQ_L(6, 3, 8) OFQ_L(6, 4, 8)
  }
#undef OFQ_L
  return OFQ_ERR_UNSUPPORTED;
}

template<typename T, int BITS>
int launch_flow_t(hipStream_t st, const LinearJob& job, const FlowPlan& plan) {
  const LinearArgs& a = job.pr[0];
  const int zmode = !a.symmetric ? kZeroAsym : (a.w_signed ? kZeroNone : kZeroSymU);
  if constexpr (BITS == 4 && TT<T>::dtype == OFQ_F16) {
    if (zmode == kZeroNone && a.group_size % 128 == 0 && a.m <= 16) {
      return launch_flow_variant<T, BITS, true, kZeroNone, true>(st, job, plan);
    }
  }
  switch (zmode) {
    case kZeroNone: return launch_flow_variant<T, BITS, true, kZeroNone>(st, job, plan);
    case kZeroSymU: return launch_flow_variant<T, BITS, false, kZeroSymU>(st, job, plan);
    default: return launch_flow_variant<T, BITS, false, kZeroAsym>(st, job, plan);
  }
}

}  // namespace
}  // namespace ofq
