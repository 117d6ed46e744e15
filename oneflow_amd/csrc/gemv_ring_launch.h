// Launch of gemv_ring (gemv_ring.h) for one T; included by one source file per T so that they compile
// side by side.
#pragma once

#include "gemv_ring.h"
#include "ofq_internal.h"

namespace ofq {
namespace {

inline RingArgs ring_args(const LinearArgs& a, const RingPlan& plan) {
  RingArgs p{};
  p.M = (int)a.m;
  p.K = (int)a.k;
  p.group_size = (int)a.group_size;
  p.gs_shift = -1;
  for (int s = 0; s < 31; ++s)
    if (((int64_t)1 << s) == a.group_size) p.gs_shift = s;
  p.rows_per_block = plan.rows_per_block;
  p.wk_shift = plan.wk_shift;
  p.phase_steps = plan.phase_steps;
  p.phases = plan.phases;
  p.m_magic = p.M == 1 ? 0u : (uint32_t)(((1ull << 32) + p.M - 1) / p.M);
  return p;
}

template<typename T, int BITS, bool SIGNED, int ZMODE, int TR, int TL>
int launch_ring_inst(hipStream_t st, const LinearJob& job, const RingPlan& plan) {
  const LinearArgs& a = job.pr[0];
  const RingArgs p = ring_args(a, plan);
  const uint16_t* x = static_cast<const uint16_t*>(a.x);
  static std::atomic<uint64_t> allowed{0}, allowed_grouped{0}, allowed_glu{0};  // devices: LDS limit raised
  if (job.glu) {
    auto kern = gemv_ring_glu<T, BITS, SIGNED, ZMODE, TR, TL>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed_glu)) return OFQ_ERR_LAUNCH;
    kern<<<plan.grid, kRingWaves * 64, plan.lds, st>>>(x, rows_mat(a), rows_mat(job.pr[1]), (int)a.n,
                                                       static_cast<uint16_t*>(job.y), job.act, p);
  } else if (job.count > 1) {
    auto kern = gemv_ring_grouped<T, BITS, SIGNED, ZMODE, TR, TL>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed_grouped)) return OFQ_ERR_LAUNCH;
    GemvGroup g{};
    fill_group(g, job.pr, job.count, plan.rows_per_block);
    kern<<<plan.grid, kRingWaves * 64, plan.lds, st>>>(g, p);
  } else {
    auto kern = gemv_ring<T, BITS, SIGNED, ZMODE, TR, TL>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed)) return OFQ_ERR_LAUNCH;
    kern<<<plan.grid, kRingWaves * 64, plan.lds, st>>>(x, rows_mat(a), (int)a.n, p);
  }
  return ofq_check_launch();
}

template<typename T, int BITS, bool SIGNED, int ZMODE>
int launch_ring_variant(hipStream_t st, const LinearJob& job, const RingPlan& plan) {
#define OFQ_L(TRV, TLV) \
  if (plan.tr == TRV && plan.tl == TLV) return launch_ring_inst<T, BITS, SIGNED, ZMODE, TRV, TLV>(st, job, plan);
  OFQ_L(8, 1) OFQ_L(8, 2) OFQ_L(8, 3) OFQ_L(8, 4)
  OFQ_L(16, 1) OFQ_L(16, 2) OFQ_L(16, 3) OFQ_L(16, 4)
#undef OFQ_L
  return OFQ_ERR_UNSUPPORTED;
}

template<typename T>
int launch_ring_t(hipStream_t st, const LinearJob& job, const RingPlan& plan) {
  const LinearArgs& a = job.pr[0];
  const int zmode = !a.symmetric ? kZeroAsym : (a.w_signed ? kZeroNone : kZeroSymU);
#define OFQ_V(B, SG, ZM)                              \
  if (a.bits == B && a.w_signed == SG && zmode == ZM) \
    return launch_ring_variant<T, B, SG, ZM>(st, job, plan);
  OFQ_V(4, true, kZeroNone)
  OFQ_V(4, false, kZeroSymU)
  OFQ_V(4, false, kZeroAsym)
  OFQ_V(8, true, kZeroNone)
  OFQ_V(8, false, kZeroSymU)
  OFQ_V(8, false, kZeroAsym)
#undef OFQ_V
  return OFQ_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace ofq
