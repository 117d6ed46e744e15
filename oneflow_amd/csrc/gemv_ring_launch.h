// Launch of gemv_ring (gemv_ring.h) for one T; included by one source file per T so that they compile
// side by side.
#pragma once

#include "gemv_ring.h"
#include "ofq_internal.h"

namespace ofq {
namespace {

struct RingPlan {
  RingArgs args;
  int tr, tl, grid;
  size_t lds;
};

inline int ring_shift(int64_t v) {
  for (int s = 0; s < 31; ++s)
    if (((int64_t)1 << s) == v) return s;
  return -1;
}

// The split of `count` problems of a's m, k and quantisation (rows: theirs; matrices: 2 for the two weights of a
// gated unit, which share blocks) or false where scales, rings and x do not fit LDS.
//
// One block per CU and round; the waves' split over tiles and K by the longest wave's turns, a turn being a
// tile's expansion and products and a step's share of reading x (about half of that).
inline bool ring_plan(const LinearArgs& a, const int64_t* rows, int count, int matrices, RingPlan* plan) {
  const int ck = a.bits == 4 ? 128 : 64, rec = ck * 2;
  const int G = (int)(a.k / a.group_size);
  const int regions = matrices * (a.symmetric ? 1 : 2);
  const int M = (int)a.m;
  const int tr = M <= 8 ? 8 : 16, sub = tr == 8 ? 2 : 1;
  const int steps = (int)((a.k + ck * sub - 1) / (ck * sub));
  constexpr int kCUs = 256, kLds = 160 * 1024;
  int64_t total = 0;
  for (int i = 0; i < count; ++i) total += rows[i];
  auto blocks_at = [&](int rpb) {
    int64_t b = 0;
    for (int i = 0; i < count; ++i) b += (rows[i] + rpb - 1) / rpb;
    return b;
  };
  for (int rounds = 1; rounds <= 512; rounds *= 2) {
    const int64_t want = (int64_t)kCUs * rounds;
    int64_t rpb64 = (total + want - 1) / want;
    if (rpb64 > 512) continue;
    int rpb = (int)rpb64 < tr ? tr : (int)rpb64;
    while (blocks_at(rpb) > want && rpb < 512) ++rpb;
    // not more tiles than the rows need: the last tile of every block full
    const int ntiles = (rpb + tr - 1) / tr;
    const int nvt = matrices * ntiles;
    const int scales = (regions * ring_scale_bytes(rpb, G) + 1023) & ~1023;
    double best = 1e30;
    for (int wk_shift = 4; wk_shift >= 0; --wk_shift) {
      const int wk = 1 << wk_shift, groups = kRingWaves >> wk_shift;
      const int tl = (nvt + groups - 1) / groups;
      if (tl > kRingMaxTiles) continue;
      const int depth = tl == 1 ? 3 : (tl == 2 ? 2 : 1);
      const int budget = kLds - scales - kRingWaves * depth * tl * 1024;
      const int step_x = sub * M * rec;
      if (budget < 1024) continue;
      int phase_steps = steps, phases = 1;
      if ((int64_t)steps * step_x > budget / 1024 * 1024) {
        phase_steps = (budget / 2 / 1024 * 1024) / step_x / wk * wk;
        if (phase_steps < wk) continue;
        phases = (steps + phase_steps - 1) / phase_steps;
        phase_steps = ((steps + phases - 1) / phases + wk - 1) / wk * wk;
        phases = (steps + phase_steps - 1) / phase_steps;
      }
      const int xbuf = (phase_steps * step_x + 1023) & ~1023;
      size_t lds = (size_t)scales + kRingWaves * depth * tl * 1024 + (size_t)xbuf * (phases > 1 ? 2 : 1);
      const size_t red = ((size_t)nvt << wk_shift) * M * 16 * 4;
      if (red > lds) lds = red;
      if (lds > kLds) continue;
      const int turns = phases == 1 ? (steps + wk - 1) / wk : phases * (phase_steps / wk);
      const double cost = turns * (tl + 0.5) + 1.0 * (phases - 1);
      if (cost < best) {
        best = cost;
        plan->tr = tr;
        plan->tl = tl;
        plan->lds = lds;
        plan->args.wk_shift = wk_shift;
        plan->args.phase_steps = phase_steps;
        plan->args.phases = phases;
      }
    }
    if (best >= 1e30) continue;
    const int64_t grid = blocks_at(rpb);
    if (grid > 0x7FFFFFFF) return false;
    plan->grid = (int)grid;
    plan->args.M = M;
    plan->args.K = (int)a.k;
    plan->args.group_size = (int)a.group_size;
    plan->args.gs_shift = ring_shift(a.group_size);
    plan->args.rows_per_block = rpb;
    plan->args.m_magic = M == 1 ? 0u : (uint32_t)(((1ull << 32) + M - 1) / M);
    return true;
  }
  return false;
}

// Where the ring is the faster one: 6000 random problems (m 1 .. 16, n 512 .. 32000, k 512 .. 14336, both types
// and widths, groups of 32, 64, 128), time of the kernels that ran before over this one's:
//   gated units                                   1.27 (5 of 100 below 1.08): two launches and the gating's
//   several linears                               1.14 (5 of 100 below 0.97)
//   one linear of more than 16 rows a block, or of whole turns of waves over short blocks   1.14
// and where it is not: one row of x of up to 4096 elements (0.87: gemv_m1_any), one linear of one 16-row tile a
// block (0.96: gemv_rows, whose requests land in registers, has nothing to balance there), and more than 8 rows
// of x that pass LDS in four parts or more (1.0, down to 0.75).
inline bool ring_preferred(const LinearArgs& a, bool one, const RingPlan& plan) {
  const RingArgs& p = plan.args;
  if (a.m > 8 && p.phases >= 4) return false;
  if (!one) return true;
  if (a.m == 1 && a.k <= 4096) return false;
  if (p.rows_per_block > 16) return true;
  const int step = (a.bits == 4 ? 128 : 64) * (plan.tr == 8 ? 2 : 1);
  const int turns = (int)((a.k + ((int64_t)step << p.wk_shift) - 1) / ((int64_t)step << p.wk_shift));
  return a.m > 1 && p.rows_per_block <= 8 && turns >= 2;
}

template<typename T, int BITS, bool SIGNED, int ZMODE, int TR, int TL>
int launch_ring_inst(hipStream_t st, const LinearJob& job, const RingPlan& plan) {
  const LinearArgs& a = job.pr[0];
  const uint16_t* x = static_cast<const uint16_t*>(a.x);
  static std::atomic<uint64_t> allowed{0}, allowed_grouped{0}, allowed_glu{0};  // devices: LDS limit raised
  if (job.glu) {
    auto kern = gemv_ring_glu<T, BITS, SIGNED, ZMODE, TR, TL>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed_glu)) return OFQ_ERR_LAUNCH;
    kern<<<plan.grid, kRingWaves * 64, plan.lds, st>>>(x, rows_mat(a), rows_mat(job.pr[1]), (int)a.n,
                                                       static_cast<uint16_t*>(job.y), job.act, plan.args);
  } else if (job.count > 1) {
    auto kern = gemv_ring_grouped<T, BITS, SIGNED, ZMODE, TR, TL>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed_grouped)) return OFQ_ERR_LAUNCH;
    GemvGroup g{};
    fill_group(g, job.pr, job.count, plan.args.rows_per_block);
    kern<<<plan.grid, kRingWaves * 64, plan.lds, st>>>(g, plan.args);
  } else {
    auto kern = gemv_ring<T, BITS, SIGNED, ZMODE, TR, TL>;
    if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, allowed)) return OFQ_ERR_LAUNCH;
    kern<<<plan.grid, kRingWaves * 64, plan.lds, st>>>(x, rows_mat(a), (int)a.n, plan.args);
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
int launch_ring_t(hipStream_t st, const LinearJob& job) {
  const LinearArgs& a = job.pr[0];
  int64_t rows[kGemvMaxProblems];
  const int lists = job.glu ? 1 : job.count;
  for (int i = 0; i < lists; ++i) rows[i] = job.pr[i].n;
  RingPlan plan;
  if (!ring_plan(a, rows, lists, job.glu ? 2 : 1, &plan) || !ring_preferred(a, job.count == 1, plan)) {
    return OFQ_ERR_UNSUPPORTED;
  }
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
