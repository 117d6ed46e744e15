// Launch of gemm_wr (gemm_wr.h) for one T; included by one source file per T so that they compile
// side by side.
#pragma once

#include "gemm_wr.h"
#include "ofq_internal.h"

namespace ofq {
namespace {

template<typename T, class MF, int BITS, bool SIGNED, int ZMODE, int TM, int WN, int KH, int NSTAGE,
         bool RAGGED, bool SPLIT>
int launch_wr_inst(hipStream_t st, const WrParams& p, int grid, size_t lds) {
  auto kern = gemm_wr<T, MF, BITS, SIGNED, ZMODE, TM, WN, KH, NSTAGE, RAGGED, SPLIT>;
  static std::atomic<uint64_t> lds_allowed{0};  // devices on which the kernel's LDS limit is raised
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, lds_allowed)) return OFQ_ERR_LAUNCH;
  kern<<<grid, WN * KH * 64, lds, st>>>(p);
  return ofq_check_launch();
}

template<typename T, class MF, int BITS, bool SIGNED, int ZMODE, int TM, int WN, int KH, int NSTAGE>
int launch_wr_cfg(hipStream_t st, const LinearArgs& a, const WrPlan& plan, float* partials) {
  constexpr size_t kStages = wr_stage_bytes<BITS, TM, WN, KH>() * NSTAGE;
  constexpr int kStepK = KH * 64;
  WrParams p;
  p.x = static_cast<const uint8_t*>(a.x);
  p.w = static_cast<const uint8_t*>(a.w);
  p.scale = static_cast<const uint16_t*>(a.scale);
  p.zero = static_cast<const uint16_t*>(a.zero);
  p.bias = static_cast<const uint16_t*>(a.bias);
  p.out = static_cast<uint16_t*>(a.out);
  p.part = partials;
  p.M = (int)a.m;
  p.N = (int)a.n;
  p.K = (int)a.k;
  p.G = (int)(a.k / a.group_size);
  p.group_magic = (uint32_t)(((1ull << 32) + a.group_size - 1) / a.group_size);
  p.group_size = (int)a.group_size;
  p.m_tiles = (int)((a.m + TM * 32 - 1) / (TM * 32));
  p.n_tiles = (int)((a.n + WN * 32 - 1) / (WN * 32));
  p.steps_total = (int)((a.k + kStepK - 1) / kStepK);
  p.steps_per_split = (p.steps_total + plan.splits - 1) / plan.splits;
  // the longest panel of scales that fits beside the stages
  const size_t per_group = (size_t)WN * 32 * 2 * (ZMODE == 2 ? 2 : 1);
  p.panel_steps = p.steps_per_split;
  size_t lds;
  for (;;) {
    int64_t groups = (int64_t)p.panel_steps * kStepK / a.group_size + 2;
    if (groups > p.G) groups = p.G;
    p.panel_groups = (int)groups;
    lds = kStages + (size_t)(groups + 1) * per_group;  // and the row of zeros
    if (lds <= 160u * 1024u) break;
    if (p.panel_steps == 1) return OFQ_ERR_UNSUPPORTED;
    p.panel_steps = (p.panel_steps + 1) / 2;
  }
  const int grid = p.m_tiles * p.n_tiles * plan.splits;
  const bool ragged = a.k % kStepK != 0;
  int rc;
  if (plan.splits == 1) {
    return ragged ? launch_wr_inst<T, MF, BITS, SIGNED, ZMODE, TM, WN, KH, NSTAGE, true, false>(st, p, grid, lds)
                  : launch_wr_inst<T, MF, BITS, SIGNED, ZMODE, TM, WN, KH, NSTAGE, false, false>(st, p, grid, lds);
  }
  rc = ragged ? launch_wr_inst<T, MF, BITS, SIGNED, ZMODE, TM, WN, KH, NSTAGE, true, true>(st, p, grid, lds)
              : launch_wr_inst<T, MF, BITS, SIGNED, ZMODE, TM, WN, KH, NSTAGE, false, true>(st, p, grid, lds);
  if (rc != OFQ_OK) return rc;
  const int tiles = ((p.M + 31) / 32) * ((p.N + 31) / 32);
  gemm_wr_fold<T><<<tiles, 256, 0, st>>>(partials, p.bias, p.out, p.M, p.N, plan.splits);
  return ofq_check_launch();
}

template<typename T, class MF, int BITS, bool SIGNED, int ZMODE>
int launch_wr_variant(hipStream_t st, const LinearArgs& a, const WrPlan& plan, float* partials) {
  switch (plan.tile) {
    case kWr32x128: return launch_wr_cfg<T, MF, BITS, SIGNED, ZMODE, 1, 4, 2, 4>(st, a, plan, partials);
    case kWr64x128: return launch_wr_cfg<T, MF, BITS, SIGNED, ZMODE, 2, 4, 2, 4>(st, a, plan, partials);
    case kWr128x256: return launch_wr_cfg<T, MF, BITS, SIGNED, ZMODE, 4, 8, 1, 4>(st, a, plan, partials);
    default: break;
  }
  if constexpr (BITS == 4) {
    switch (plan.tile) {
      case kWr96x128: return launch_wr_cfg<T, MF, BITS, SIGNED, ZMODE, 3, 4, 2, 4>(st, a, plan, partials);
      case kWr192x256: return launch_wr_cfg<T, MF, BITS, SIGNED, ZMODE, 6, 8, 1, 4>(st, a, plan, partials);
      default: break;
    }
  }
  return OFQ_ERR_UNSUPPORTED;
}

template<typename T, class MF>
int launch_wr_t(hipStream_t st, const LinearArgs& a, const WrPlan& plan, float* partials) {
  const int zmode = !a.symmetric ? 2 : (a.w_signed ? 0 : 1);
#define OFQ_V(B, SG, ZM)                              \
  if (a.bits == B && a.w_signed == SG && zmode == ZM) \
    return launch_wr_variant<T, MF, B, SG, ZM>(st, a, plan, partials);
  OFQ_V(4, true, 0)
  OFQ_V(4, false, 1)
  OFQ_V(4, false, 2)
  OFQ_V(8, true, 0)
  OFQ_V(8, false, 1)
  OFQ_V(8, false, 2)
#undef OFQ_V
  return OFQ_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace ofq
