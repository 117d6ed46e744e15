// Launch of gemv_ring_mt (gemv_ring_mt.h) for one T; included by one source file per T and width of codes so that
// they compile side by side.
#pragma once

#include "gemv_ring_mt.h"
#include "ofq_internal.h"

namespace ofq {
namespace {

inline RingMtArgs ring_mt_args(const LinearArgs& a, const RingMtPlan& plan) {
  RingMtArgs p{};
  p.M = (int)a.m;
  p.K = (int)a.k;
  p.group_size = (int)a.group_size;
  p.gs_shift = -1;
  for (int s = 0; s < 31; ++s)
    if (((int64_t)1 << s) == a.group_size) p.gs_shift = s;
  p.rows_per_block = plan.rows_per_block;
  p.wk = plan.wk;
  p.depth = plan.depth;
  p.buffers = plan.buffers;
  p.phases = plan.phases;
  p.m_magic = (uint32_t)(((1ull << 32) + p.M - 1) / p.M);
  return p;
}

template<typename T, int BITS, bool SIGNED, int ZMODE, int MT, int TL>
int launch_ring_mt_inst(hipStream_t st, const LinearJob& job, const RingMtPlan& plan) {
  const LinearArgs& a = job.pr[0];
  const RingMtArgs p = ring_mt_args(a, plan);
  const uint16_t* x = static_cast<const uint16_t*>(a.x);
  static std::atomic<uint64_t> allowed{0}, allowed_grouped{0}, allowed_glu{0};  // devices: LDS limit raised
  if (job.glu) {
    auto kern = gemv_ring_mt_glu<T, BITS, SIGNED, ZMODE, MT, TL>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed_glu)) return OFQ_ERR_LAUNCH;
    kern<<<plan.grid, kRingWaves * 64, plan.lds, st>>>(x, rows_mat(a), rows_mat(job.pr[1]), (int)a.n,
                                                       static_cast<uint16_t*>(job.y), job.act, p);
  } else if (job.count > 1) {
    auto kern = gemv_ring_mt_grouped<T, BITS, SIGNED, ZMODE, MT, TL>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed_grouped)) return OFQ_ERR_LAUNCH;
    GemvGroup g{};
    fill_group(g, job.pr, job.count, plan.rows_per_block);
    kern<<<plan.grid, kRingWaves * 64, plan.lds, st>>>(g, p);
  } else {
    auto kern = gemv_ring_mt<T, BITS, SIGNED, ZMODE, MT, TL>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed)) return OFQ_ERR_LAUNCH;
    kern<<<plan.grid, kRingWaves * 64, plan.lds, st>>>(x, rows_mat(a), (int)a.n, p);
  }
  return ofq_check_launch();
}

template<typename T, int BITS, bool SIGNED, int ZMODE>
int launch_ring_mt_variant(hipStream_t st, const LinearJob& job, const RingMtPlan& plan) {
  const int mt = (int)((job.pr[0].m + 15) / 16);
#define OFQ_L(MTV, TLV) \
  if (mt == MTV && plan.tl == TLV) return launch_ring_mt_inst<T, BITS, SIGNED, ZMODE, MTV, TLV>(st, job, plan);
  OFQ_L(2, 1) OFQ_L(2, 2) OFQ_L(2, 3)
  OFQ_L(3, 1) OFQ_L(3, 2) OFQ_L(3, 3)
  OFQ_L(4, 1) OFQ_L(4, 2) OFQ_L(4, 3)
#undef OFQ_L
  return OFQ_ERR_UNSUPPORTED;
}

template<typename T, int BITS>
int launch_ring_mt_t(hipStream_t st, const LinearJob& job, const RingMtPlan& plan) {
  const LinearArgs& a = job.pr[0];
  if (!a.symmetric) return launch_ring_mt_variant<T, BITS, false, kZeroAsym>(st, job, plan);
  return a.w_signed ? launch_ring_mt_variant<T, BITS, true, kZeroNone>(st, job, plan)
                    : launch_ring_mt_variant<T, BITS, false, kZeroSymU>(st, job, plan);
}

}  // namespace
}  // namespace ofq
