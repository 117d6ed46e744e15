// Launch of gemv_rows_mt (gemv_rows.h) for one T; included by one source file per T so that they compile
// side by side.
#pragma once

#include "gemv_rows.h"
#include "ofq_internal.h"

namespace ofq {
namespace {

inline int mt_shift(int64_t v) {
  for (int s = 0; s < 31; ++s)
    if (((int64_t)1 << s) == v) return s;
  return -1;
}

template<typename T, int BITS, bool SIGNED, int ZMODE, int NW, int MT, int NTL>
int launch_rows_mt_inst(hipStream_t st, const LinearJob& job, const RowsMtPlan& p) {
  const LinearArgs& a = job.pr[0];
  const int shift = mt_shift(a.group_size);
  const uint16_t* x = static_cast<const uint16_t*>(a.x);
  static std::atomic<uint64_t> allowed{0}, allowed_grouped{0};  // devices: the kernel's LDS limit is raised
  if (job.count > 1) {
    auto kern = gemv_rows_mt_grouped<T, BITS, SIGNED, ZMODE, NW, MT, NTL>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed_grouped)) return OFQ_ERR_LAUNCH;
    GemvGroup g{};
    fill_group(g, job.pr, job.count, p.rows_per_block);
    kern<<<p.grid, NW * 64, p.lds, st>>>(g, (int)a.m, (int)a.k, (int)a.group_size, shift, p.rows_per_block,
                                        p.panel_chunks, p.panel_groups);
    return ofq_check_launch();
  }
  auto kern = gemv_rows_mt<T, BITS, SIGNED, ZMODE, NW, MT, NTL>;
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed)) return OFQ_ERR_LAUNCH;
  const RowsMat mat = rows_mat(a);
  kern<<<p.grid, NW * 64, p.lds, st>>>(x, mat.w, mat.scale, mat.zero, mat.bias, mat.out, (int)a.m, (int)a.n,
                                      (int)a.k, (int)a.group_size, shift, p.rows_per_block,
                                      p.panel_chunks, p.panel_groups);
  return ofq_check_launch();
}

template<typename T, int BITS, bool SIGNED, int ZMODE, int NW, int MT, int NTL>
int launch_rows_mt_glu_inst(hipStream_t st, const LinearJob& job, const RowsMtPlan& p) {
  const LinearArgs& a = job.pr[0];
  auto kern = gemv_rows_mt_glu<T, BITS, SIGNED, ZMODE, NW, MT, NTL>;
  static std::atomic<uint64_t> lds_allowed{0};  // devices on which the kernel's LDS limit is raised
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, lds_allowed)) return OFQ_ERR_LAUNCH;
  kern<<<p.grid, NW * 64, p.lds, st>>>(static_cast<const uint16_t*>(a.x), rows_mat(a), rows_mat(job.pr[1]),
                                      static_cast<uint16_t*>(job.y), job.act, (int)a.m, (int)a.n, (int)a.k,
                                      (int)a.group_size, mt_shift(a.group_size), p.rows_per_block,
                                      p.panel_chunks, p.panel_groups);
  return ofq_check_launch();
}

template<typename T, int NW, int MT>
int launch_rows_mt_t(hipStream_t st, const LinearJob& job, const RowsMtPlan& p) {
  const LinearArgs& a = job.pr[0];
  const int zmode = !a.symmetric ? kZeroAsym : (a.w_signed ? kZeroNone : kZeroSymU);
#define OFQ_R(B, SG, ZM)                                                                          \
  if (a.bits == B && a.w_signed == SG && zmode == ZM) {                                           \
    if (job.glu) {                                                                                \
      return p.rows_per_block <= 16 ? launch_rows_mt_glu_inst<T, B, SG, ZM, NW, MT, 1>(st, job, p) \
                                    : launch_rows_mt_glu_inst<T, B, SG, ZM, NW, MT, 2>(st, job, p); \
    }                                                                                             \
    return p.rows_per_block <= 16   ? launch_rows_mt_inst<T, B, SG, ZM, NW, MT, 1>(st, job, p)    \
           : p.rows_per_block <= 32 ? launch_rows_mt_inst<T, B, SG, ZM, NW, MT, 2>(st, job, p)    \
                                    : launch_rows_mt_inst<T, B, SG, ZM, NW, MT, 4>(st, job, p);   \
  }
  OFQ_R(4, true, kZeroNone)
  OFQ_R(4, false, kZeroSymU)
  OFQ_R(4, false, kZeroAsym)
  OFQ_R(8, true, kZeroNone)
  OFQ_R(8, false, kZeroSymU)
  OFQ_R(8, false, kZeroAsym)
#undef OFQ_R
  return OFQ_ERR_UNSUPPORTED;
}

template<typename T>
int launch_rows_mt_plan(hipStream_t st, const LinearJob& job, const RowsMtPlan& p) {
  switch ((int)((job.pr[0].m + 15) / 16)) {
    case 2: return launch_rows_mt_t<T, 12, 2>(st, job, p);
    case 3: return launch_rows_mt_t<T, 8, 3>(st, job, p);
    default: return launch_rows_mt_t<T, 8, 4>(st, job, p);
  }
}

}  // namespace
}  // namespace ofq
