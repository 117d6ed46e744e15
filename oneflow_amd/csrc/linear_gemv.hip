// fused_linear_with_groupwise_quantized_weight, decode side (m <= 16), for gfx950, plus the
// any-shape fallback and the op's C entry point.
//
// Semantics (oneflow/user/kernels/groupwise_quantization_kernels.cu:582-642, :760-839):
//   w~[n,k] = T(T(q[n,k]) * scale[n,g]) + zero[n,g]   (both operations round to T)
//   out[m,n] = T( sum_k x[m,k] * w~[n,k]  (fp32 accumulation)  + float(bias[n]) )
//
// Decode kernel.  The reference launches one 128-thread block per output element and so streams
// the weights m times.  Here the m <= 16 rows of x ride along as the second operand of a
// 16x16x32 MFMA whose first dimension is 16 weight rows, so the weights are read from HBM exactly
// once whatever m is, and the k-reduction happens inside the matrix core instead of in a
// cross-lane tree:
//   - a block owns 16 consecutive weight rows and all of K; its waves take K in interleaved
//     chunks of 128 (4-bit) / 64 (8-bit) elements, i.e. one 128-bit load per lane covering
//     16 rows x 64 bytes;
//   - lane (r = lane%16, kb = lane/16) loads 16 bytes of row r; its 32 (16) codes feed the
//     "k-slot kb" of 4 (2) MFMAs.  The MFMA sums over k-slots, so any assignment of k to
//     (slot, element) is valid as long as the x operand uses the same one;
//   - int4 -> fp16 without conversions: (word & 0x000F000F) | 0x64006400 is the half2
//     (1024+q_lo, 1024+q_hi); the nibbles 4 bits up give 1024+16q.  One packed add (or fma by
//     1/16) recovers the codes exactly; an int8 container is first xor-ed with 0x88888888 to
//     turn two's complement nibbles into offset binary.  The codes come out pairwise
//     (e1,e5),(e0,e4),(e3,e7),(e2,e6) and x is permuted to match with four v_perm_b32;
//   - w~ is then formed exactly as the reference does (packed fp16 multiply by the group scale,
//     packed add of the zero term), bit-compatible with groupwise_dequantize -- in every kernel
//     but the fp16 fast path for symmetric 4-bit codes in an int8 container (gemv_w4s_f16 and
//     gemv_w4p_f16 with EXACT = false), which scales the exact fp32 group sum instead and never
//     rounds q*scale to fp16 (~3e-4 rel-L2 from the composition);
//   - partial sums of the waves are combined through LDS, bias is added in fp32, one rounding
//     to T.
#include <atomic>
#include "gemv_kernels.h"
#include "gemv_flow.h"
#include "gemv_ring.h"
#include "gemv_rows.h"
#include "ofq_device.h"
#include "ofq_internal.h"

namespace ofq {
namespace {

// ---- any shape, any grouping: one wave per weight row and up to MT rows of x ----------------
// The fallback for what the streaming kernels do not take (k off their chunk grid, odd group
// sizes).  A wave owns weight row n, its lanes walk k (two adjacent codes of a byte per step for
// 4-bit weights, so that a wave's requests are 64 consecutive bytes of codes), every element is
// dequantised once with the reference's roundings and meets the rows m0 .. m0+MT-1 of x;
// indices are 32-bit (the entry point bounds m*k, n*k and m*n by 2^31).
template<typename T, int BITS, bool SIGNED, int MT>
__global__ void __launch_bounds__(256)
linear_generic(const typename TT<T>::storage* __restrict__ x, const uint8_t* __restrict__ w,
               const typename TT<T>::storage* __restrict__ scale,
               const typename TT<T>::storage* __restrict__ zero,
               const typename TT<T>::storage* __restrict__ bias,
               typename TT<T>::storage* __restrict__ out, int M, int N, int K, int group_dim,
               int group_size, int symmetric) {
  constexpr int E = BITS == 4 ? 2 : 1;
  const int lane = threadIdx.x & 63;
  const int n = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int m0 = (int)blockIdx.y * MT;
  if (n >= N) return;
  float acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = 0.f;
  auto zero_term = [&](float s, int si) -> float {
    if (!symmetric) return TT<T>::load(zero + si);
    if (SIGNED) return 0.f;
    return TT<T>::round(-(float)((1 << (BITS - 1)) - 1) * s);
  };
  auto element = [&](int k, float s, float z) {
    const float q = (float)code_at<BITS, SIGNED>(w, (int64_t)n * K + k);
    const float wv = TT<T>::round(TT<T>::round(q * s) + z);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if (m0 + i < M) acc[i] = __builtin_fmaf(TT<T>::load(x + (m0 + i) * K + k), wv, acc[i]);
    }
  };
  if (group_dim == 1) {
    // group by group: scale and zero are the same for the whole wave (one broadcast request per
    // group instead of one per element, no division per element).  Items (group, step of 64*E
    // elements within it) are taken four at a time with all their requests issued before any is
    // used: a wave walks its row alone, and one memory round trip per item would bound it.
    const int G = K / group_size;
    const int spg = (group_size + 64 * E - 1) / (64 * E);  // steps per group
    const int items = G * spg;
    constexpr int B = 4;
    for (int it0 = 0; it0 < items; it0 += B) {
      float sv[B], zv[B];
      int kk[B][E];
      bool ok[B][E];
      int code[B][E];
      float xv[B][E][MT];
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const int it = it0 + b < items ? it0 + b : items - 1;
        const int gi = it / spg;  // (the same for every lane)
        const int st = it - gi * spg;
        const int si = n * G + gi;
        sv[b] = TT<T>::load(scale + si);
        zv[b] = zero_term(sv[b], si);
        const int kend = (gi + 1) * group_size;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const int k = gi * group_size + st * 64 * E + lane * E + e;
          ok[b][e] = it0 + b < items && k < kend;
          kk[b][e] = ok[b][e] ? k : 0;
          code[b][e] = code_at<BITS, SIGNED>(w, (int64_t)n * K + kk[b][e]);
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            xv[b][e][i] = TT<T>::load(x + (m0 + i < M ? m0 + i : m0) * K + kk[b][e]);
          }
        }
      }
#pragma unroll
      for (int b = 0; b < B; ++b) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const float wv = TT<T>::round(TT<T>::round((float)code[b][e] * sv[b]) + zv[b]);
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            if (ok[b][e] && m0 + i < M) acc[i] = __builtin_fmaf(xv[b][e][i], wv, acc[i]);
          }
        }
      }
    }
  } else {
    const int srow = (n / group_size) * K;
    for (int k0 = lane * E; k0 < K; k0 += 64 * E) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int k = k0 + e;
        if (k < K) {
          const float s = TT<T>::load(scale + srow + k);
          element(k, s, zero_term(s, srow + k));
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const float sum = wave_reduce(acc[i], OpSum());
    if (lane == 0 && m0 + i < M) {
      float r = sum;
      if (bias != nullptr) r += TT<T>::load(bias + n);
      TT<T>::store(out + (m0 + i) * N + n, r);
    }
  }
}

template<typename T>
int launch_generic_t(hipStream_t st, const LinearArgs& a) {
  typedef typename TT<T>::storage S;
  if (a.group_size > 0x7FFFFFFF) return OFQ_ERR_UNSUPPORTED;
#define OFQ_G1(B, SG, MTV)                                                                   \
  {                                                                                          \
    dim3 grid((unsigned)((a.n + 3) / 4), (unsigned)((a.m + MTV - 1) / MTV));                 \
    linear_generic<T, B, SG, MTV><<<grid, 256, 0, st>>>(                                     \
        static_cast<const S*>(a.x), static_cast<const uint8_t*>(a.w),                        \
        static_cast<const S*>(a.scale), static_cast<const S*>(a.zero),                       \
        static_cast<const S*>(a.bias), static_cast<S*>(a.out), (int)a.m, (int)a.n, (int)a.k, \
        a.group_dim, (int)a.group_size, a.symmetric ? 1 : 0);                                \
    return ofq_check_launch();                                                               \
  }
#define OFQ_G(B, SG)                                                                         \
  if (a.bits == B && a.w_signed == SG) {                                                     \
    if (a.m == 1) OFQ_G1(B, SG, 1)                                                           \
    if (a.m <= 4) OFQ_G1(B, SG, 4)                                                           \
    OFQ_G1(B, SG, 8)                                                                         \
  }
  OFQ_G(4, false) OFQ_G(4, true) OFQ_G(8, false) OFQ_G(8, true)
#undef OFQ_G
#undef OFQ_G1
  return OFQ_ERR_UNSUPPORTED;
}

inline int ilog2_exact(int64_t v) {
  if (v <= 0 || (v & (v - 1)) != 0) return -1;
  int s = 0;
  while ((1LL << s) < v) ++s;
  return s;
}

// ---- fast path launcher (gemv_w4s_f16) ------------------------------------------------------
template<int NW, bool STAGED>
int launch_w4s_inst(hipStream_t st, const LinearArgs& a, size_t lds, int cpg_shift) {
  auto kern = gemv_w4s_f16<NW, 2, STAGED>;
  if (lds > 64 * 1024) return OFQ_ERR_UNSUPPORTED;
  const int grid = (int)((a.n + 15) / 16);
  kern<<<grid, NW * 64, lds, st>>>(static_cast<const f16*>(a.x), static_cast<const uint8_t*>(a.w),
                                  static_cast<const f16*>(a.scale),
                                  static_cast<const f16*>(a.bias), static_cast<f16*>(a.out),
                                  (int)a.m, (int)a.n, (int)a.k, (int)a.group_size, cpg_shift);
  return ofq_check_launch();
}

bool w4s_supported(const LinearArgs& a) {
  return a.t_dtype == OFQ_F16 && a.bits == 4 && a.w_signed && a.symmetric && a.group_dim == 1
         && a.m >= 1 && a.m <= 16 && a.k % 128 == 0 && a.group_size % 128 == 0
         && a.k <= (1 << 20) && a.n <= 0x7FFFFFFF - 16;
}

// Row-balanced kernel: grid = a whole number of blocks per CU (or one 16-row tile per block when
// n is small), rows_per_block <= 64.
template<int NW, bool EXACT, bool SIGNED, int ZMODE, bool TILED = false, int PH = 1>
int launch_w4p_inst(hipStream_t st, const LinearArgs& a, int grid, int rows_per_block, size_t lds,
                    int cpg_shift) {
  auto kern = gemv_w4p_f16<NW, 1, EXACT, SIGNED, ZMODE, TILED, PH>;
  static std::atomic<uint64_t> lds_allowed{0};  // devices on which the kernel's LDS limit is raised
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, lds_allowed)) return OFQ_ERR_LAUNCH;
  kern<<<grid, NW * 64, lds, st>>>(static_cast<const f16*>(a.x), static_cast<const uint8_t*>(a.w),
                                  static_cast<const f16*>(a.scale),
                                  static_cast<const f16*>(a.zero),
                                  static_cast<const f16*>(a.bias), static_cast<f16*>(a.out),
                                  (int)a.m, (int)a.n, (int)a.k, (int)a.group_size, cpg_shift,
                                  rows_per_block);
  return ofq_check_launch();
}

// 4-bit codes, fp16, groups along K in multiples of 128: what the row-balanced kernel takes
bool w4p_supported(const LinearArgs& a) {
  return a.t_dtype == OFQ_F16 && a.bits == 4 && a.group_dim == 1 && a.m >= 1 && a.m <= 16
         && a.k % 128 == 0 && a.group_size % 128 == 0 && a.k <= (1 << 20)
         && a.n <= 0x7FFFFFFF - 16 && (a.symmetric || !a.w_signed);
}

// The row split of the row-balanced kernel, a function of n alone (the tile-major weight copy is
// laid out by it): one block per CU of a 256-CU part when that keeps a block within 64 rows (a
// single 16-row tile per block when n is small), else two, else as many 64-row blocks as it takes.
void w4p_row_split(int64_t n, int64_t* grid_out, int* rows_per_block_out) {
  constexpr int kCUs = 256;
  const int64_t max_rows = 16 * kW4pMaxTiles;
  int64_t grid = kCUs;
  if ((n + grid - 1) / grid > max_rows) grid = 2 * kCUs;
  if ((n + grid - 1) / grid > max_rows) grid = (n + max_rows - 1) / max_rows;
  int rpb = (int)((n + grid - 1) / grid);
  if (rpb < 16) rpb = 16;
  *grid_out = (n + rpb - 1) / rpb;
  *rows_per_block_out = rpb;
}

// OFQ_ERR_UNSUPPORTED when the shape does not fit the row-balanced kernel
int launch_w4p(hipStream_t st, const LinearArgs& a, int cpg_shift, bool tiled) {
  constexpr int kCUs = 256;
  int64_t grid;
  int rpb;
  w4p_row_split(a.n, &grid, &rpb);
  const bool two_per_cu = grid > kCUs;
  const int nw = two_per_cu ? 8 : 16;
  // one thread folds one output of the block
  if ((int64_t)((rpb + 15) / 16) * a.m * 16 > nw * 64) return OFQ_ERR_UNSUPPORTED;
  const bool exact = !(a.symmetric && a.w_signed);
  const size_t lds_cap = (two_per_cu ? 80u : 160u) * 1024u;
  size_t lds = gemv_w4p_lds_bytes(nw, (int)a.m, (int)a.k, (int)a.group_size, rpb, exact,
                                  !a.symmetric);
  if (a.m * a.k / 16 > (int64_t)kGemvMaxUnits * nw * 64 || lds > lds_cap) {
    // m * k beyond one staging of x: two to four stagings, each of an equal part of the chunk
    // pairs of a row (one block per CU only)
    if (nw != 16) return OFQ_ERR_UNSUPPORTED;
    int phases = 0;
    for (int ph = 2; ph <= 4 && phases == 0; ++ph) {
      const int64_t part_units = a.m * gemv_w4p_phase_chunks((int)a.k, ph) * 8;
      lds = gemv_w4p_lds_bytes(nw, (int)a.m, (int)a.k, (int)a.group_size, rpb, exact,
                               !a.symmetric, 1, ph);
      if (part_units <= (int64_t)kGemvMaxUnits * nw * 64 && lds <= lds_cap) phases = ph;
    }
    if (phases == 0) return OFQ_ERR_UNSUPPORTED;
#define OFQ_W4PN(TL, PHV)                                                                    \
  if (tiled == TL && phases == PHV) {                                                        \
    if (!exact)                                                                              \
      return launch_w4p_inst<16, false, true, kZeroNone, TL, PHV>(st, a, (int)grid, rpb,     \
                                                                  lds, cpg_shift);           \
    if (a.symmetric)                                                                         \
      return launch_w4p_inst<16, true, false, kZeroSymU, TL, PHV>(st, a, (int)grid, rpb,     \
                                                                  lds, cpg_shift);           \
    return launch_w4p_inst<16, true, false, kZeroAsym, TL, PHV>(st, a, (int)grid, rpb, lds,  \
                                                                cpg_shift);                  \
  }
    OFQ_W4PN(false, 2) OFQ_W4PN(true, 2) OFQ_W4PN(false, 3) OFQ_W4PN(true, 3)
    OFQ_W4PN(false, 4) OFQ_W4PN(true, 4)
#undef OFQ_W4PN
  }
#define OFQ_W4P(NWV, TL)                                                                     \
  if (nw == NWV && tiled == TL) {                                                            \
    if (!exact)                                                                              \
      return launch_w4p_inst<NWV, false, true, kZeroNone, TL>(st, a, (int)grid, rpb, lds,    \
                                                              cpg_shift);                    \
    if (a.symmetric)                                                                         \
      return launch_w4p_inst<NWV, true, false, kZeroSymU, TL>(st, a, (int)grid, rpb, lds,    \
                                                              cpg_shift);                    \
    return launch_w4p_inst<NWV, true, false, kZeroAsym, TL>(st, a, (int)grid, rpb, lds,      \
                                                            cpg_shift);                      \
  }
  OFQ_W4P(16, false) OFQ_W4P(8, false) OFQ_W4P(16, true) OFQ_W4P(8, true)
#undef OFQ_W4P
  return OFQ_ERR_UNSUPPORTED;
}

// ---- natural-order row-balanced kernel (gemv_rows): fp16 / bf16, 4- and 8-bit ----------------
template<typename T, int BITS, bool SIGNED, int ZMODE, int NW, bool STAGED>
int launch_rows_inst(hipStream_t st, const LinearArgs& a, int grid, int rows_per_block,
                     size_t lds, int gs_shift) {
  auto kern = gemv_rows<T, BITS, SIGNED, ZMODE, NW, STAGED>;
  static std::atomic<uint64_t> lds_allowed{0};  // devices on which the kernel's LDS limit is raised
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, lds_allowed)) return OFQ_ERR_LAUNCH;
  kern<<<grid, NW * 64, lds, st>>>(
      static_cast<const uint16_t*>(a.x), static_cast<const uint8_t*>(a.w),
      static_cast<const uint16_t*>(a.scale), static_cast<const uint16_t*>(a.zero),
      static_cast<const uint16_t*>(a.bias), static_cast<uint16_t*>(a.out), (int)a.m, (int)a.n,
      (int)a.k, (int)a.group_size, gs_shift, rows_per_block);
  return ofq_check_launch();
}

bool rows_supported(const LinearArgs& a) {
  if (a.t_dtype != OFQ_F16 && a.t_dtype != OFQ_BF16) return false;
  if (a.bits != 4 && a.bits != 8) return false;
  const int lk = a.bits == 4 ? 32 : 16;  // elements behind a lane's 16 bytes of codes
  return a.group_dim == 1 && a.m >= 1 && a.m <= 16 && a.k % lk == 0
         && a.group_size % lk == 0 && a.k <= (1 << 20) && a.n <= 0x7FFFFFFF - 16
         && (a.symmetric || !a.w_signed);
}

// The split of gemv_ring for a job, or false where scales, rings and x do not fit LDS.
//
// One block per CU and round; the waves' split over tiles and K by the longest wave's turns, a turn being a
// tile's expansion and products and a step's share of reading x (about half of that).
bool ring_plan(const LinearJob& job, RingPlan* plan) {
  const LinearArgs& a = job.pr[0];
  const int lists = job.glu ? 1 : job.count, matrices = job.glu ? 2 : 1;
  const int ck = a.bits == 4 ? 128 : 64, rec = ck * 2;
  const int G = (int)(a.k / a.group_size);
  const int regions = matrices * (a.symmetric ? 1 : 2);
  const int M = (int)a.m;
  const int tr = M <= 8 ? 8 : 16, sub = tr == 8 ? 2 : 1;
  const int steps = (int)((a.k + ck * sub - 1) / (ck * sub));
  constexpr int kCUs = 256, kLds = 160 * 1024;
  int64_t total = 0;
  for (int i = 0; i < lists; ++i) total += job.pr[i].n;
  auto blocks_at = [&](int rpb) {
    int64_t b = 0;
    for (int i = 0; i < lists; ++i) b += (job.pr[i].n + rpb - 1) / rpb;
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
        plan->wk_shift = wk_shift;
        plan->phase_steps = phase_steps;
        plan->phases = phases;
      }
    }
    if (best >= 1e30) continue;
    const int64_t grid = blocks_at(rpb);
    if (grid > 0x7FFFFFFF) return false;
    plan->grid = (int)grid;
    plan->rows_per_block = rpb;
    return true;
  }
  return false;
}

}  // namespace

namespace {

// The split of gemv_flow for a job, or false where more than a block per CU or LDS would be needed: eight waves, or
// six where eight leave no room.
bool flow_plan(const LinearJob& job, FlowPlan* plan) {
  const LinearArgs& a = job.pr[0];
  const int lists = job.glu ? 1 : job.count, matrices = job.glu ? 2 : 1;
  const int G = (int)(a.k / a.group_size);
  const int regions = matrices * (a.symmetric ? 1 : 2);
  const int mx = a.m <= 8 ? 1 : a.m <= 16 ? 2 : a.m <= 32 ? 4 : 6;
  const int max_rows = job.glu ? 48 : mx == 1 ? 96 : mx == 2 ? 80 : 64;
  int64_t total = 0;
  for (int i = 0; i < lists; ++i) total += job.pr[i].n;
  auto blocks_at = [&](int rpb) {
    int64_t b = 0;
    for (int i = 0; i < lists; ++i) b += (job.pr[i].n + rpb - 1) / rpb;
    return b;
  };
  int rpb = total > 256 * max_rows ? max_rows + 1 : (int)((total + 255) / 256);
  if (rpb < 16) rpb = 16;
  while (rpb <= max_rows && blocks_at(rpb) > 256) ++rpb;
  if (rpb <= max_rows) {
    const int tl = (rpb + 15) / 16;
    const size_t scales = (size_t)(regions * ring_scale_bytes(rpb, G) + 1023) & ~(size_t)1023;
    const int step = flow_x_ops(a.bits, mx) + flow_chunks(a.bits, mx) * tl * matrices;
    for (int nw = 8; nw >= (mx > 2 ? 8 : 6); nw -= 2) {
      size_t lds = scales + (size_t)nw * step * 1024;
      const size_t red = (size_t)nw * (size_t)a.m * (tl * matrices * 16 + 4) * 4;
      if (red > lds) lds = red;
      if (lds > 160 * 1024) continue;
      plan->grid = (int)blocks_at(rpb);
      plan->rows_per_block = rpb;
      plan->mx = mx;
      plan->tl = tl;
      plan->nw = nw;
      plan->tiled = 0;
      plan->lds = lds;
      return true;
    }
  }
  return false;
}

}  // namespace

// Whether gemv_flow takes a job, and how; asked after the row-per-wave kernels of one row of x.  Time over that of the
// kernels which would run instead, on 260 random jobs (m 1 .. 16, n 512 .. 32000, k 512 .. 14336, all types, widths and
// groups of 32, 64, 128, weights from HBM):
//   several linears                                       0.88 (one row of x and more than 48 rows a block: 1.05)
//   one linear of 9 to 16 rows of x                       0.88
//   one linear of up to 8, more than 8 rows a block       0.93 (0.78 to 1.08)
//   gated units of 9 to 16 rows of x                      0.94 (0.57 where x has to pass gemv_w4p_f16_glu in parts)
//   gated units of up to 8 on one tile, or two that are   0.90 (0.71 to 1.02)
//   filled to three quarters
// and where it is not the faster one:
//   more than one round of blocks                         1.0 to 1.25
//   blocks of up to 8 rows, up to 8 rows of x             1.0 to 1.28 (half of every tile is nobody's)
//   other gated units of up to 8 rows of x                1.03 (to 1.13; gemv_ring's 8-row tiles), on fp16 4-bit groups
//                                                         of whole chunks and up to 4 rows 1.02 (gemv_w4p_f16_glu)
//   bf16 4-bit, more than 64 rows a block                 1.02: bound by the expansion either way
//   one linear of up to 4 rows of x on fp16 4-bit groups  1.06 to 1.14 (gemv_w4s_f16)
//   of whole chunks, up to 16 rows a block
// On 149 other jobs: 0.94, 6 more than 3 % longer, 1.13 at worst (8 x 2 x 3584 x 1280 fp16 4-bit with a zero point).
// A tile-major copy of a weight (fp16, 4 bits, groups of whole chunks) is asked by the same rule, so that the two calls
// give the same bits; its blocks have up to 64 rows, as many as here.
bool gemv_flow_choice(const LinearJob& job, FlowPlan* plan) {
  const LinearArgs& a = job.pr[0];
  for (int i = 0; i < job.count; ++i) {
    const LinearArgs& b = job.pr[i];
    if (!rows_supported(b) || b.t_dtype != a.t_dtype || b.bits != a.bits || b.w_signed != a.w_signed
        || b.symmetric != a.symmetric || b.group_size != a.group_size || b.m != a.m || b.k != a.k) {
      return false;
    }
  }
  int64_t rows = 0;  // of a block
  for (int i = 0; i < (job.glu ? 1 : job.count); ++i) rows += job.pr[i].n;
  rows = (rows + 255) / 256;
  const bool bf16_4 = a.t_dtype == OFQ_BF16 && a.bits == 4;
  const bool late = a.t_dtype == OFQ_F16 && a.bits == 4 && a.symmetric && a.w_signed && a.group_size % 128 == 0;
  if (job.glu) {
    if (rows > 48) return false;
    if (a.m <= 8 && !(rows <= 16 || (rows >= 25 && rows <= 32) || (rows >= 44 && a.bits == 8))) return false;
    if (a.m <= 4 && late) return false;
  } else if (job.count > 1) {
    if (rows > 80 || (rows > 48 && a.m == 1)) return false;
  } else {
    if (rows > (a.m > 8 || bf16_4 || w4p_supported(a) ? 64 : 96) || (a.m <= 8 && rows <= 8)) return false;
    if (late && a.m <= 4 && rows <= 16) return false;
  }
  return flow_plan(job, plan);
}

namespace {

int launch_flow_by(hipStream_t st, const LinearJob& job, const FlowPlan& plan) {
  const bool four = job.pr[0].bits == 4;
  if (job.pr[0].t_dtype == OFQ_BF16) {
    return four ? launch_gemv_flow_bf16_b4(st, job, plan) : launch_gemv_flow_bf16_b8(st, job, plan);
  }
  return four ? launch_gemv_flow_f16_b4(st, job, plan) : launch_gemv_flow_f16_b8(st, job, plan);
}
int launch_flow(hipStream_t st, const LinearJob& job) {
  FlowPlan plan;
  return gemv_flow_choice(job, &plan) ? launch_flow_by(st, job, plan) : OFQ_ERR_UNSUPPORTED;
}

}  // namespace

// Whether gemv_ring takes a job, and how.  (The plan comes last: its loops run for every call, and small calls are
// bound by the host: 3 x 1560 x 1024 bf16 5.7 us with the plan, 5.3 before it.)
// Time against the kernels that would run instead, on 12 400 random jobs (m 1 .. 16, n 512 .. 32000, k 512 .. 14336,
// both types and widths, groups of 32, 64, 128, weights from HBM):
//   gated units                                          0.75, none of 3000 longer: two launches and the gating's
//   several linears                                      0.91, 28 of 2500 more than 3 % longer, 1.09 at worst
//   one linear of more than 16 rows a block, or of whole turns of waves over short blocks
//                                                        0.86, 109 of 4700 more than 3 % longer, 1.15 at worst
// and where it is not the faster one:
//   one row of x of up to 4096 elements                  1.15 (gemv_m1_any)
//   one linear of one 16-row tile a block                1.04 (gemv_rows, whose requests land in registers, has nothing
//                                                        to balance there)
//   up to 8 rows of x, blocks of whole 16-row tiles:     one linear of 25 to 32 rows a block and 2 to 4 turns of
//                                                        gemv_rows' waves 1.03 (0.9 to 1.25); several of 25 to 32 rows
//                                                        and 2 turns 1.03 (0.95 to 1.1), of 9 to 16 rows, up to 3
//                                                        rows of x and 2 turns and more 1.01 (to 1.08)
//   more than 8 rows of x that pass LDS in four parts or more 1.0, up to 1.33
bool gemv_ring_choice(const LinearJob& job, RingPlan* plan) {
  const LinearArgs& a = job.pr[0];
  for (int i = 0; i < job.count; ++i) {
    const LinearArgs& b = job.pr[i];
    if (!rows_supported(b) || b.t_dtype != a.t_dtype || b.bits != a.bits || b.w_signed != a.w_signed
        || b.symmetric != a.symmetric || b.group_size != a.group_size || b.m != a.m || b.k != a.k) {
      return false;
    }
  }
  int64_t rows = 0;  // of a block
  for (int i = 0; i < (job.glu ? 1 : job.count); ++i) rows += job.pr[i].n;
  rows = (rows + 255) / 256;
  const int tiles8 = (int)((rows + 7) / 8);
  const int64_t turns = (a.k - 1) / (16 * (a.bits == 4 ? 128 : 64)) + 1;  // of gemv_rows' waves
  // (fp16 with 4-bit codes and no zero point has the shortest expansion, in gemv_ring's own order)
  const bool whole = a.m <= 8 && !(a.t_dtype == OFQ_F16 && a.bits == 4 && a.symmetric);
  if (job.count == 1) {
    if (a.m == 1 && a.k <= 4096) return false;
    if (rows <= 16 && !(a.m > 1 && a.m <= 8 && rows <= 8 && turns > 2)) return false;
    if (whole && tiles8 == 4 && turns >= 2 && turns <= 4) return false;
  } else if (!job.glu && whole && ((tiles8 == 2 && turns >= 2 && a.m <= 3) || (tiles8 == 4 && turns == 2))) {
    return false;
  }
  return ring_plan(job, plan) && !(a.m > 8 && plan->phases >= 4);
}

namespace {

int launch_ring(hipStream_t st, const LinearJob& job) {
  RingPlan plan;
  if (!gemv_ring_choice(job, &plan)) return OFQ_ERR_UNSUPPORTED;
  return job.pr[0].t_dtype == OFQ_BF16 ? launch_gemv_ring_bf16(st, job, plan) : launch_gemv_ring_f16(st, job, plan);
}

template<typename T, int NW>
int launch_rows_t(hipStream_t st, const LinearArgs& a, int grid, int rpb, size_t lds,
                  bool staged) {
  const int gs_shift = ilog2_exact(a.group_size);
  const int zmode = !a.symmetric ? kZeroAsym : (a.w_signed ? kZeroNone : kZeroSymU);
#define OFQ_R(B, SG, ZM)                                              \
  if (a.bits == B && a.w_signed == SG && zmode == ZM)                 \
    return staged ? launch_rows_inst<T, B, SG, ZM, NW, true>(st, a, grid, rpb, lds, gs_shift) \
                  : launch_rows_inst<T, B, SG, ZM, NW, false>(st, a, grid, rpb, lds, gs_shift);
  OFQ_R(4, true, kZeroNone)
  OFQ_R(4, false, kZeroSymU)
  OFQ_R(4, false, kZeroAsym)
  OFQ_R(8, true, kZeroNone)
  OFQ_R(8, false, kZeroSymU)
  OFQ_R(8, false, kZeroAsym)
#undef OFQ_R
  return OFQ_ERR_UNSUPPORTED;
}

// OFQ_ERR_UNSUPPORTED when x does not fit the block's registers and LDS
int launch_rows(hipStream_t st, const LinearArgs& a) {
  {
    const int rc = launch_ring(st, LinearJob{&a, 1, false, nullptr, 0});
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  constexpr int kCUs = 256;
  const int64_t max_rows = 16 * kRowsMaxTiles;
  int64_t grid = kCUs;
  if ((a.n + grid - 1) / grid > max_rows) grid = 2 * kCUs;
  if ((a.n + grid - 1) / grid > max_rows) grid = (a.n + max_rows - 1) / max_rows;
  int rpb = (int)((a.n + grid - 1) / grid);
  if (rpb < 16) rpb = 16;
  grid = (a.n + rpb - 1) / rpb;
  const bool two_per_cu = grid > kCUs;
  const int nw = two_per_cu ? 8 : 16;
  const size_t cap = (two_per_cu ? 80u : 160u) * 1024u;
  // x goes to LDS when it fits there and in the staging registers; else it is read from L2
  bool staged = a.m * a.k / 8 <= (int64_t)kRowsMaxUnits * nw * 64;
  // bf16 with 4-bit codes and a zero term is bound by the vector unit (eleven instructions per
  // element pair); staging more than 64 KB of x adds to that (11008 x 4096 at 16 rows: 16.0
  // against 15.2 us), where the 8-bit and the symmetric variants gain from it (fp16 W8: 14.2
  // against 15.3 us)
  if (a.t_dtype == OFQ_BF16 && a.bits == 4 && !(a.symmetric && a.w_signed)
      && a.m * a.k * 2 > 65536) {
    staged = false;
  }
  size_t lds = gemv_rows_lds_bytes(nw, (int)a.m, (int)a.k, (int)a.group_size, rpb,
                                   !a.symmetric, staged);
  if (staged && lds > cap) {
    staged = false;
    lds = gemv_rows_lds_bytes(nw, (int)a.m, (int)a.k, (int)a.group_size, rpb, !a.symmetric,
                              false);
  }
  if (lds > cap) return OFQ_ERR_UNSUPPORTED;
  if (a.t_dtype == OFQ_BF16) {
    return nw == 16 ? launch_rows_t<bf16, 16>(st, a, (int)grid, rpb, lds, staged)
                    : launch_rows_t<bf16, 8>(st, a, (int)grid, rpb, lds, staged);
  }
  return nw == 16 ? launch_rows_t<f16, 16>(st, a, (int)grid, rpb, lds, staged)
                  : launch_rows_t<f16, 8>(st, a, (int)grid, rpb, lds, staged);
}

int launch_w4s(hipStream_t st, const LinearArgs& a) {
  const int64_t tiles = (a.n + 15) / 16;
  const int npairs = (int)((a.k / 128 + 1) / 2);
  const int cpg_shift = ilog2_exact(a.group_size / 128);
  // waves per block: as many as still let every block be resident at once (<= 24 waves per CU on
  // 256 CUs), so the kernel runs as a single round of blocks; never more than there are pairs
  // and never fewer than fold the block's m * 16 outputs with one thread each
  const int nw_min = a.m > 8 ? 4 : 2;
  int nw = 16;
  while (nw > nw_min && (tiles * nw > 6144 || nw > npairs)) nw >>= 1;
  const int nt = nw * 64;
  const int64_t nunits = a.m * a.k / 16;
  bool staged = nunits <= (int64_t)kGemvMaxUnits * nt;
  size_t lds = gemv_w4s_lds_bytes(nw, staged, (int)a.m, (int)a.k, (int)a.group_size);
  if (staged && lds > 48 * 1024) {
    staged = false;
    lds = gemv_w4s_lds_bytes(nw, false, (int)a.m, (int)a.k, (int)a.group_size);
  }
  // More than one 16-row tile per CU, or an x too large to stage per 16 rows: the row-balanced
  // kernel (equal bytes per block, x staged once per block) is the faster one.
  if (tiles > 256 || !staged) {
    int rc = launch_w4p(st, a, cpg_shift, false);
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
    // x too large for either staged kernel: the natural-order kernel reads x from L2 once per
    // block, the one below once per 16 rows
    if (!staged) {
      rc = launch_rows(st, a);
      if (rc != OFQ_ERR_UNSUPPORTED) return rc;
    }
  }
#define OFQ_W4S(NWV)                                                                   \
  if (nw == NWV)                                                                       \
    return staged ? launch_w4s_inst<NWV, true>(st, a, lds, cpg_shift)                  \
                  : launch_w4s_inst<NWV, false>(st, a, lds, cpg_shift);
  OFQ_W4S(16) OFQ_W4S(8) OFQ_W4S(4) OFQ_W4S(2)
#undef OFQ_W4S
  return OFQ_ERR_UNSUPPORTED;
}

template<int BITS, bool SIGNED, int ZMODE>
int launch_gemv_variant(hipStream_t st, const LinearArgs& a) {
  constexpr int CH = BITS == 4 ? 128 : 64;
  const int nchunks = (int)(a.k / CH);
  const int grid = (int)((a.n + 15) / 16);
  const int gs_shift = ilog2_exact(a.group_size);
  const f16* x = static_cast<const f16*>(a.x);
  const uint8_t* w = static_cast<const uint8_t*>(a.w);
  const f16* sc = static_cast<const f16*>(a.scale);
  const f16* ze = static_cast<const f16*>(a.zero);
  const f16* bi = static_cast<const f16*>(a.bias);
  f16* out = static_cast<f16*>(a.out);
  // waves per block: enough to spread K, few enough that every wave has >= 2 chunks
  if (nchunks >= 64) {
    gemv_f16_mfma<BITS, SIGNED, ZMODE, 16, 2><<<grid, 16 * 64, 0, st>>>(
        x, w, sc, ze, bi, out, (int)a.m, (int)a.n, (int)a.k, (int)a.group_size, gs_shift);
  } else if (nchunks >= 16) {
    gemv_f16_mfma<BITS, SIGNED, ZMODE, 8, 4><<<grid, 8 * 64, 0, st>>>(
        x, w, sc, ze, bi, out, (int)a.m, (int)a.n, (int)a.k, (int)a.group_size, gs_shift);
  } else {
    gemv_f16_mfma<BITS, SIGNED, ZMODE, 4, 2><<<grid, 4 * 64, 0, st>>>(
        x, w, sc, ze, bi, out, (int)a.m, (int)a.n, (int)a.k, (int)a.group_size, gs_shift);
  }
  return ofq_check_launch();
}

// ---- 16 < m <= 64: several tiles of x per weight tile -----------------------------------------
// Rows per block (of each matrix) and blocks: one round of blocks, one per CU, if a block's rows are then at
// most the kernel's weight tiles.
constexpr int kMtGluTiles = 2;  // of each of the two weights
void rows_mt_split(const LinearJob& job, int* rpb, int64_t* grid) {
  constexpr int kCUs = 256;
  const int lists = job.glu ? 1 : job.count;
  const int max_rows = 16 * (job.glu ? kMtGluTiles : kRowsMaxTiles);
  int64_t total = 0;
  for (int i = 0; i < lists; ++i) total += job.pr[i].n;
  auto blocks_at = [&](int r) {
    int64_t b = 0;
    for (int i = 0; i < lists; ++i) b += (job.pr[i].n + r - 1) / r;
    return b;
  };
  int64_t rows = (total + kCUs - 1) / kCUs;
  if (rows < 16) rows = 16;
  if (job.glu && rows > max_rows) {  // whole rounds
    const int64_t rounds = (rows + max_rows - 1) / max_rows;
    rows = (total + kCUs * rounds - 1) / (kCUs * rounds);
  }
  if (rows > max_rows) rows = max_rows;
  int r = (int)rows;
  while (r < max_rows && blocks_at(r) > kCUs && total <= (int64_t)kCUs * max_rows) ++r;
  *rpb = r;
  *grid = blocks_at(r);
}

// The split of gemv_ring_mt, or false where scales, rings and x do not fit LDS.  One block per CU and round; the
// workers' split over tiles and K by the longest wave's steps: of a step, each tile's expansion and products, and
// what it takes whatever it has of them, x among it.
bool ring_mt_plan(const LinearJob& job, RingMtPlan* plan) {
  const LinearArgs& a = job.pr[0];
  constexpr int kCUs = 256, kLds = 160 * 1024, kMaxTl = 3, kWorkers = 12;
  const int lists = job.glu ? 1 : job.count, matrices = job.glu ? 2 : 1;
  const int ck = a.bits == 4 ? 128 : 64;
  const int64_t G = a.k / a.group_size;
  const int regions = matrices * (a.symmetric ? 1 : 2);
  const int64_t steps = (a.k + ck - 1) / ck;
  const int64_t step_x = a.m * ck * 2;
  if (G * 2 * 16 > kLds) return false;
  int64_t total = 0;
  for (int i = 0; i < lists; ++i) total += job.pr[i].n;
  auto blocks_at = [&](int64_t r) {
    int64_t b = 0;
    for (int i = 0; i < lists; ++i) b += (job.pr[i].n + r - 1) / r;
    return b;
  };
  for (int64_t rounds = 1; rounds <= 512; rounds *= 2) {
    const int64_t want = kCUs * rounds;
    int64_t rpb = (total + want - 1) / want;
    if (rpb > 16 * kMaxTl * kWorkers) continue;
    if (rpb < 16) rpb = 16;
    while (blocks_at(rpb) > want && rpb < 16 * kMaxTl * kWorkers) ++rpb;
    const int64_t nvt = matrices * ((rpb + 15) / 16);
    const int64_t scales = (regions * ((rpb * G * 2 + 16 + 15) & ~15) + 1023) & ~(int64_t)1023;
    double best = 1e30;
    for (int wk = kWorkers; wk >= 1; --wk) {
      if (kWorkers % wk != 0) continue;
      const int64_t tl = (nvt + kWorkers / wk - 1) / (kWorkers / wk);
      if (tl > kMaxTl) continue;
      const int64_t xbuf = (wk * step_x + 1023) & ~(int64_t)1023;
      if (xbuf > 64 * 1024) continue;  // kRingMtCopies
      const int most = tl == 1 ? 3 : (tl == 2 ? 2 : 1);
      int buffers = 4, depth = 0;
      for (; buffers >= 2; --buffers) {
        const int64_t left = kLds - scales - buffers * xbuf;
        depth = left < 0 ? 0 : (int)(left / (kWorkers * tl * 1024));
        depth = depth < most ? depth : most;
        if (depth >= (most < 2 || buffers == 2 ? 1 : 2)) break;
      }
      if (buffers < 2) continue;
      const size_t red = (size_t)nvt * wk * a.m * 64;
      if (red > kLds) continue;
      const int64_t phases = (steps + wk - 1) / wk;
      const double cost = phases * (tl + 0.2 + 0.1 * ((a.m + 15) / 16) + 0.5);
      if (cost < best) {
        best = cost;
        plan->tl = (int)tl;
        plan->wk = wk;
        plan->depth = depth;
        plan->buffers = buffers;
        plan->phases = (int)phases;
        plan->lds = (size_t)(scales + kWorkers * depth * tl * 1024 + buffers * xbuf);
        if (red > plan->lds) plan->lds = red;
      }
    }
    if (best >= 1e30) continue;
    const int64_t grid = blocks_at(rpb);
    if (grid > 0x7FFFFFFF) return false;
    plan->grid = (int)grid;
    plan->rows_per_block = (int)rpb;
    return true;
  }
  return false;
}

int launch_ring_mt(hipStream_t st, const LinearJob& job, const RingMtPlan& plan) {
  const LinearArgs& a = job.pr[0];
  if (a.t_dtype == OFQ_BF16) {
    return a.bits == 4 ? launch_gemv_ring_mt_bf16_b4(st, job, plan) : launch_gemv_ring_mt_bf16_b8(st, job, plan);
  }
  return a.bits == 4 ? launch_gemv_ring_mt_f16_b4(st, job, plan) : launch_gemv_ring_mt_f16_b8(st, job, plan);
}

int launch_rows_mt(hipStream_t st, const LinearJob& job) {
  const LinearArgs& a = job.pr[0];
  RowsMtPlan p;
  int64_t grid;
  rows_mt_split(job, &p.rows_per_block, &grid);
  if (grid > 0x7FFFFFFF) return OFQ_ERR_UNSUPPORTED;
  p.grid = (int)grid;
  // 12 waves for two tiles of x, 8 for three and four (the x buffers and the registers of the
  // requests in flight)
  const int mt = (int)((a.m + 15) / 16);
  const int nw = mt == 2 ? 12 : 8;
  // the longest panel of scales that fits beside the x buffers, in whole turns of the waves
  const int ck = a.bits == 4 ? 128 : 64;
  const int turn = 2 * nw;
  int turns = (int)(((a.k + ck - 1) / ck + turn - 1) / turn);
  for (;; --turns) {
    if (turns < 1) return OFQ_ERR_UNSUPPORTED;
    p.panel_chunks = turns * turn;
    const int64_t groups = ((int64_t)p.panel_chunks * ck) / a.group_size + 2;
    const int64_t all = a.k / a.group_size;
    p.panel_groups = (int)(groups < all ? groups : all);
    p.lds = gemv_rows_mt_lds_bytes(nw, mt, a.bits, p.rows_per_block, p.panel_groups, !a.symmetric,
                                   job.glu ? 2 : 1);
    if (p.lds <= 160u * 1024u) break;
  }
  return a.t_dtype == OFQ_BF16 ? launch_gemv_mt_bf16(st, job, p) : launch_gemv_mt_f16(st, job, p);
}

// ---- fp32 activations -------------------------------------------------------------------------
template<int BITS, bool SIGNED, int ZMODE>
int launch_rows_f32_inst(hipStream_t st, const LinearArgs& a, const float* x, float* out, int m,
                         int grid, int rows_per_block, size_t lds) {
  auto kern = gemv_rows_f32<BITS, SIGNED, ZMODE, 16>;
  static std::atomic<uint64_t> lds_allowed{0};  // devices on which the kernel's LDS limit is raised
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, lds_allowed)) return OFQ_ERR_LAUNCH;
  kern<<<grid, 16 * 64, lds, st>>>(x, static_cast<const uint8_t*>(a.w),
                                  static_cast<const float*>(a.scale),
                                  static_cast<const float*>(a.zero),
                                  static_cast<const float*>(a.bias), out, m, (int)a.n, (int)a.k,
                                  (int)a.group_size, ilog2_exact(a.group_size), rows_per_block);
  return ofq_check_launch();
}

bool rows_f32_supported(const LinearArgs& a) {
  if (a.t_dtype != OFQ_F32 || (a.bits != 4 && a.bits != 8)) return false;
  const int ck = a.bits == 4 ? 128 : 64;
  return a.group_dim == 1 && a.m >= 1 && a.k % ck == 0 && a.group_size % (ck / 4) == 0
         && a.k <= (1 << 20) && a.n <= 0x7FFFFFFF - 16 && (a.symmetric || !a.w_signed);
}

// any m: 16 rows of x per pass over the weights
int launch_rows_f32(hipStream_t st, const LinearArgs& a) {
  constexpr int kCUs = 256;
  const int64_t max_rows = 16 * kRowsMaxTiles;
  int64_t grid = kCUs;
  if ((a.n + grid - 1) / grid > max_rows) grid = (a.n + max_rows - 1) / max_rows;
  int rpb = (int)((a.n + grid - 1) / grid);
  if (rpb < 16) rpb = 16;
  grid = (a.n + rpb - 1) / rpb;
  const size_t lds =
      gemv_rows_f32_lds_bytes(16, (int)a.k, (int)a.group_size, rpb, !a.symmetric);
  if (lds > 160u * 1024u) return OFQ_ERR_UNSUPPORTED;
  const int zmode = !a.symmetric ? kZeroAsym : (a.w_signed ? kZeroNone : kZeroSymU);
  for (int64_t m0 = 0; m0 < a.m; m0 += 16) {
    const int m = (int)(a.m - m0 < 16 ? a.m - m0 : 16);
    const float* x = static_cast<const float*>(a.x) + m0 * a.k;
    float* out = static_cast<float*>(a.out) + m0 * a.n;
    int rc = OFQ_ERR_UNSUPPORTED;
#define OFQ_R(B, SG, ZM)                                              \
  if (a.bits == B && a.w_signed == SG && zmode == ZM)                 \
    rc = launch_rows_f32_inst<B, SG, ZM>(st, a, x, out, m, (int)grid, rpb, lds);
    OFQ_R(4, true, kZeroNone)
    OFQ_R(4, false, kZeroSymU)
    OFQ_R(4, false, kZeroAsym)
    OFQ_R(8, true, kZeroNone)
    OFQ_R(8, false, kZeroSymU)
    OFQ_R(8, false, kZeroAsym)
#undef OFQ_R
    if (rc != OFQ_OK) return rc;
  }
  return OFQ_OK;
}

// ---- several problems, one launch -------------------------------------------------------------
template<typename T, int BITS, bool SIGNED, int ZMODE, int NW, bool STAGED>
int launch_rows_grouped_inst(hipStream_t st, const GemvGroup& g, int grid, int m, int k,
                             int group_size, int rows_per_block, size_t lds) {
  auto kern = gemv_rows_grouped<T, BITS, SIGNED, ZMODE, NW, STAGED>;
  static std::atomic<uint64_t> lds_allowed{0};  // devices on which the kernel's LDS limit is raised
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, lds_allowed)) return OFQ_ERR_LAUNCH;
  kern<<<grid, NW * 64, lds, st>>>(g, m, k, group_size, ilog2_exact(group_size), rows_per_block);
  return ofq_check_launch();
}

template<typename T, int NW, bool STAGED>
int launch_rows_grouped_t(hipStream_t st, const LinearArgs& a, const GemvGroup& g, int grid,
                          int rpb, size_t lds) {
  const int zmode = !a.symmetric ? kZeroAsym : (a.w_signed ? kZeroNone : kZeroSymU);
#define OFQ_R(B, SG, ZM)                                                           \
  if (a.bits == B && a.w_signed == SG && zmode == ZM)                              \
    return launch_rows_grouped_inst<T, B, SG, ZM, NW, STAGED>(st, g, grid, (int)a.m, (int)a.k, \
                                                              (int)a.group_size, rpb, lds);
  OFQ_R(4, true, kZeroNone)
  OFQ_R(4, false, kZeroSymU)
  OFQ_R(4, false, kZeroAsym)
  OFQ_R(8, true, kZeroNone)
  OFQ_R(8, false, kZeroSymU)
  OFQ_R(8, false, kZeroAsym)
#undef OFQ_R
  return OFQ_ERR_UNSUPPORTED;
}

template<int NW, bool EXACT, bool SIGNED, int ZMODE, int PH = 1>
int launch_w4p_grouped_inst(hipStream_t st, const GemvGroup& g, int grid, int m, int k,
                            int group_size, int rows_per_block, size_t lds) {
  auto kern = gemv_w4p_f16_grouped<NW, EXACT, SIGNED, ZMODE, PH>;
  static std::atomic<uint64_t> lds_allowed{0};  // devices on which the kernel's LDS limit is raised
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, lds_allowed)) return OFQ_ERR_LAUNCH;
  kern<<<grid, NW * 64, lds, st>>>(g, m, k, group_size, ilog2_exact(group_size / 128),
                                  rows_per_block);
  return ofq_check_launch();
}

// the smallest common rows_per_block (>= 16, <= max_rows) whose blocks fit one resident round:
// 256 blocks of 16 waves, else 512 of 8; returns the grid size
int64_t grouped_split(const LinearArgs* pr, int count, int max_rows, int* rpb_out) {
  constexpr int kCUs = 256;
  int64_t n_total = 0;
  for (int i = 0; i < count; ++i) n_total += pr[i].n;
  auto blocks_at = [&](int rpb) {
    int64_t b = 0;
    for (int i = 0; i < count; ++i) b += (pr[i].n + rpb - 1) / rpb;
    return b;
  };
  int rpb = (int)((n_total + kCUs - 1) / kCUs);
  if (rpb < 16) rpb = 16;
  while (rpb < max_rows && blocks_at(rpb) > kCUs) ++rpb;
  if (rpb > max_rows || blocks_at(rpb) > kCUs) {
    rpb = (int)((n_total + 2 * kCUs - 1) / (2 * kCUs));
    if (rpb < 16) rpb = 16;
    while (rpb < max_rows && blocks_at(rpb) > 2 * kCUs) ++rpb;
  }
  if (rpb > max_rows) rpb = max_rows;
  *rpb_out = rpb;
  return blocks_at(rpb);
}

// fp16, 4-bit codes, groups in multiples of 128: the kernel of the single-problem fast path
int launch_w4p_grouped(hipStream_t st, const LinearArgs* pr, int count) {
  const LinearArgs& a = pr[0];
  int rpb = 0;
  const int64_t grid = grouped_split(pr, count, 16 * kW4pMaxTiles, &rpb);
  if (grid > 0x7FFFFFFF) return OFQ_ERR_UNSUPPORTED;
  const bool two_per_cu = grid > 256;
  const int nw = two_per_cu ? 8 : 16;
  if ((int64_t)((rpb + 15) / 16) * a.m * 16 > nw * 64) return OFQ_ERR_UNSUPPORTED;
  const bool exact = !(a.symmetric && a.w_signed);
  const size_t lds_cap = (two_per_cu ? 80u : 160u) * 1024u;
  size_t lds = gemv_w4p_lds_bytes(nw, (int)a.m, (int)a.k, (int)a.group_size, rpb, exact,
                                  !a.symmetric);
  // x beyond one staging: two stagings, each of half the chunk pairs of a row
  const bool two_stagings = a.m * a.k / 16 > (int64_t)kGemvMaxUnits * nw * 64 || lds > lds_cap;
  if (two_stagings) {
    lds = gemv_w4p_lds_bytes(nw, (int)a.m, (int)a.k, (int)a.group_size, rpb, exact, !a.symmetric,
                             1, 2);
    const int64_t half_units = a.m * gemv_w4p_phase_chunks((int)a.k, 2) * 8;
    if (half_units > (int64_t)kGemvMaxUnits * nw * 64 || lds > lds_cap) return OFQ_ERR_UNSUPPORTED;
  }
  GemvGroup g{};
  fill_group(g, pr, count, rpb);
#define OFQ_W4PG(NWV, PHV)                                                                   \
  if (nw == NWV && two_stagings == (PHV == 2)) {                                             \
    if (!exact)                                                                              \
      return launch_w4p_grouped_inst<NWV, false, true, kZeroNone, PHV>(                      \
          st, g, (int)grid, (int)a.m, (int)a.k, (int)a.group_size, rpb, lds);                \
    if (a.symmetric)                                                                         \
      return launch_w4p_grouped_inst<NWV, true, false, kZeroSymU, PHV>(                      \
          st, g, (int)grid, (int)a.m, (int)a.k, (int)a.group_size, rpb, lds);                \
    return launch_w4p_grouped_inst<NWV, true, false, kZeroAsym, PHV>(                        \
        st, g, (int)grid, (int)a.m, (int)a.k, (int)a.group_size, rpb, lds);                  \
  }
  OFQ_W4PG(16, 1) OFQ_W4PG(8, 1) OFQ_W4PG(16, 2) OFQ_W4PG(8, 2)
#undef OFQ_W4PG
  return OFQ_ERR_UNSUPPORTED;
}

template<int NW, bool EXACT, bool SIGNED, int ZMODE, int PH = 1>
int launch_w4p_glu_inst(hipStream_t st, const LinearArgs& a, const GluArgs& glu, int grid,
                        int rows_per_block, size_t lds) {
  auto kern = gemv_w4p_f16_glu<NW, EXACT, SIGNED, ZMODE, PH>;
  static std::atomic<uint64_t> lds_allowed{0};  // devices on which the kernel's LDS limit is raised
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, lds_allowed)) return OFQ_ERR_LAUNCH;
  kern<<<grid, NW * 64, lds, st>>>(static_cast<const f16*>(a.x), static_cast<const uint8_t*>(a.w),
                                  static_cast<const f16*>(a.scale),
                                  static_cast<const f16*>(a.zero),
                                  static_cast<const f16*>(a.bias), static_cast<f16*>(a.out), glu,
                                  (int)a.m, (int)a.n, (int)a.k, (int)a.group_size,
                                  ilog2_exact(a.group_size / 128), rows_per_block);
  return ofq_check_launch();
}

int launch_w4p_glu(hipStream_t st, const LinearArgs& a, const LinearArgs& g, void* y, int act) {
  if (!w4p_supported(a) || !w4p_supported(g)) return OFQ_ERR_UNSUPPORTED;
  constexpr int kCUs = 256;
  const bool exact = !(a.symmetric && a.w_signed);
  // A block walks the same rows of both weights.  First choice: up to 64 rows of each per block,
  // so that n = 11008 is one block of 16 waves per CU as in the plain linear (43 rows, three
  // tiles per weight); that doubles the per-(tile, wave) sums in LDS, so with many rows of x it
  // may not fit, and then a block owns at most 32 rows of each weight (two blocks per CU).
  int64_t grid = 0;
  int rpb = 0, nw = 0;
  size_t lds = 0;
  bool two_stagings = false, fits = false;
  for (int tiles_per_weight = kW4pMaxTiles; tiles_per_weight >= kW4pMaxTiles / 2 && !fits;
       tiles_per_weight -= kW4pMaxTiles / 2) {
    const int64_t max_rows = 16 * tiles_per_weight;
    grid = kCUs;
    if ((a.n + grid - 1) / grid > max_rows) grid = 2 * kCUs;
    if ((a.n + grid - 1) / grid > max_rows) grid = (a.n + max_rows - 1) / max_rows;
    rpb = (int)((a.n + grid - 1) / grid);
    if (rpb < 16) rpb = 16;
    grid = (a.n + rpb - 1) / rpb;
    const bool two_per_cu = grid > kCUs;
    nw = two_per_cu ? 8 : 16;
    // one thread folds one output of the block (per weight)
    if ((int64_t)((rpb + 15) / 16) * a.m * 16 > nw * 64) continue;
    const size_t lds_cap = (two_per_cu ? 80u : 160u) * 1024u;
    lds = gemv_w4p_lds_bytes(nw, (int)a.m, (int)a.k, (int)a.group_size, rpb, exact, !a.symmetric,
                             2);
    // x beyond one staging (8 rows of 4096 next to the sums of two weights): two stagings
    two_stagings = a.m * a.k / 16 > (int64_t)kGemvMaxUnits * nw * 64 || lds > lds_cap;
    if (two_stagings) {
      lds = gemv_w4p_lds_bytes(nw, (int)a.m, (int)a.k, (int)a.group_size, rpb, exact,
                               !a.symmetric, 2, 2);
      const int64_t half_units = a.m * gemv_w4p_phase_chunks((int)a.k, 2) * 8;
      if (half_units > (int64_t)kGemvMaxUnits * nw * 64 || lds > lds_cap) continue;
    }
    fits = true;
  }
  if (!fits) return OFQ_ERR_UNSUPPORTED;
  GluArgs glu;
  glu.w2 = static_cast<const uint8_t*>(g.w);
  glu.scale2 = static_cast<const f16*>(g.scale);
  glu.zero2 = static_cast<const f16*>(g.zero);
  glu.bias2 = static_cast<const f16*>(g.bias);
  glu.out2 = static_cast<f16*>(g.out);
  glu.y = static_cast<f16*>(y);
  glu.act = act;
#define OFQ_W4PGLU(NWV, PHV)                                                                   \
  if (nw == NWV && two_stagings == (PHV == 2)) {                                               \
    if (!exact)                                                                                \
      return launch_w4p_glu_inst<NWV, false, true, kZeroNone, PHV>(st, a, glu, (int)grid, rpb, \
                                                                   lds);                       \
    if (a.symmetric)                                                                           \
      return launch_w4p_glu_inst<NWV, true, false, kZeroSymU, PHV>(st, a, glu, (int)grid, rpb, \
                                                                   lds);                       \
    return launch_w4p_glu_inst<NWV, true, false, kZeroAsym, PHV>(st, a, glu, (int)grid, rpb,   \
                                                                 lds);                         \
  }
  OFQ_W4PGLU(16, 1) OFQ_W4PGLU(8, 1) OFQ_W4PGLU(16, 2) OFQ_W4PGLU(8, 2)
#undef OFQ_W4PGLU
  return OFQ_ERR_UNSUPPORTED;
}

}  // namespace

int launch_gemv_glu(hipStream_t st, const LinearArgs& a, const LinearArgs& g, void* y, int act) {
  int rc = launch_gemv_m1_glu(st, a, g, y, act);
  if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  if (g.n != a.n || g.k != a.k || g.m != a.m || g.x != a.x) return OFQ_ERR_UNSUPPORTED;
  const LinearArgs both[2] = {a, g};
  {
    const int rc = launch_flow(st, LinearJob{both, 2, true, y, act});
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  rc = launch_w4p_glu(st, a, g, y, act);
  if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  return launch_ring(st, LinearJob{both, 2, true, y, act});
}

int launch_gemv_grouped(hipStream_t st, const LinearArgs* pr, int count) {
  if (count < 1 || count > kGemvMaxProblems) return OFQ_ERR_UNSUPPORTED;
  {
    const int rc = launch_gemv_m1_grouped(st, pr, count);
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  const LinearArgs& a = pr[0];
  bool all_w4p = true;
  for (int i = 0; i < count; ++i) {
    const LinearArgs& b = pr[i];
    if (!rows_supported(b)) return OFQ_ERR_UNSUPPORTED;
    if (b.t_dtype != a.t_dtype || b.bits != a.bits || b.w_signed != a.w_signed
        || b.symmetric != a.symmetric || b.group_size != a.group_size || b.m != a.m
        || b.k != a.k) {
      return OFQ_ERR_UNSUPPORTED;
    }
    all_w4p = all_w4p && w4p_supported(b);
  }
  {
    const int rc = launch_flow(st, LinearJob{pr, count, false, nullptr, 0});
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  if (all_w4p) {
    const int rc = launch_w4p_grouped(st, pr, count);
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  if (count > 1) {
    const int rc = launch_ring(st, LinearJob{pr, count, false, nullptr, 0});
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  int rpb = 0;
  const int64_t grid = grouped_split(pr, count, 16 * kRowsMaxTiles, &rpb);
  if (grid > 0x7FFFFFFF) return OFQ_ERR_UNSUPPORTED;
  const bool two_per_cu = grid > 256;
  const int nw = two_per_cu ? 8 : 16;
  const size_t cap = (two_per_cu ? 80u : 160u) * 1024u;
  bool staged = a.m * a.k / 8 <= (int64_t)kRowsMaxUnits * nw * 64;
  size_t lds = gemv_rows_lds_bytes(nw, (int)a.m, (int)a.k, (int)a.group_size, rpb, !a.symmetric,
                                   staged);
  if (staged && lds > cap) {
    staged = false;
    lds = gemv_rows_lds_bytes(nw, (int)a.m, (int)a.k, (int)a.group_size, rpb, !a.symmetric,
                              false);
  }
  if (lds > cap) return OFQ_ERR_UNSUPPORTED;
  GemvGroup g{};
  fill_group(g, pr, count, rpb);
#define OFQ_RG(TT_, NWV)                                                                   \
  return staged ? launch_rows_grouped_t<TT_, NWV, true>(st, a, g, (int)grid, rpb, lds)     \
                : launch_rows_grouped_t<TT_, NWV, false>(st, a, g, (int)grid, rpb, lds)
  if (a.t_dtype == OFQ_BF16) {
    if (nw == 16) { OFQ_RG(bf16, 16); }
    OFQ_RG(bf16, 8);
  }
  if (nw == 16) { OFQ_RG(f16, 16); }
  OFQ_RG(f16, 8);
#undef OFQ_RG
}

namespace {

bool gemv_mt_supported(const LinearArgs& a) {
  // beyond 64 rows the weights would be walked twice and the tiled GEMM with K slices is faster
  if (a.m <= 16 || a.m > 64) return false;
  LinearArgs b = a;
  b.m = 16;  // the same shape rules as the decode kernel
  return rows_supported(b) && a.n * a.k <= 0x7FFFFFFFLL * 8;
}

}  // namespace

// Expected time of gemv_rows_mt in us, within 27 % of the measured one for 98 of 100 shapes (those of
// wr_plan_us with up to 64 rows).  A round of blocks starts and ends (4.25, the scales, the output); a turn of
// a block's waves over their chunks takes a part per tile of weights expanded, one per row of weights
// read and one per row of x read (every block reads all of x, from L2).
static double rows_mt_us(const LinearJob& job) {
  const LinearArgs& a = job.pr[0];
  const bool b4 = a.bits == 4;
  const int nw = a.m <= 32 ? 12 : 8;
  const int ck = b4 ? 128 : 64;
  int rows;
  int64_t blocks;
  rows_mt_split(job, &rows, &blocks);
  const int matrices = job.glu ? 2 : 1;
  const int grid = (int)blocks, tiles = matrices * ((rows + 15) / 16);
  int64_t outputs = 0;
  for (int i = 0; i < job.count; ++i) outputs += a.m * job.pr[i].n;
  rows *= matrices;
  const int turns = (int)(((a.k + ck - 1) / ck + nw - 1) / nw);
  // bf16 with a zero point has the longest conversion
  const double longer = b4 && a.t_dtype == OFQ_BF16 && !(a.symmetric && a.w_signed) ? 1.21 : 1.0;
  const double turn_us = b4 ? 0.26 + (0.50 * tiles + 0.20 * rows / 16) * longer + 0.0020 * a.m * nw
                            : 0.10 + 0.26 * tiles + 0.31 * rows / 16 + 0.0009 * a.m * nw;
  const int rest = grid % 256, rounds = (grid + 255) / 256;
  const double scales = (double)a.k / a.group_size * rows * (a.symmetric ? 1 : 2);
  return rounds * (4.25 + 1.4 / 4096 * scales) - 0.8 + 2.3e-6 * outputs
         + turns * turn_us * (grid / 256 + (rest != 0 ? 0.83 + 0.17 * rest / 256 : 0.0));
}

// Expected time of gemv_ring_mt in us, within 18 % of the measured one for 96 of 100 (500 random problems of 17 to
// 64 rows: linears of 512 to 32000 x 512 to 14336, several of a layer, gated units).  A round of blocks starts
// and ends; a phase (a step of every wave) takes a part per tile of its waves expanded and one per row
// of x that every wave reads from LDS.
static double ring_mt_us(const LinearJob& job, const RingMtPlan& plan) {
  const LinearArgs& a = job.pr[0];
  const bool b4 = a.bits == 4;
  const int matrices = job.glu ? 2 : 1;
  const int rounds = (plan.grid + 255) / 256;
  const double tiles = matrices * ((plan.rows_per_block + 15) / 16);
  double outputs = 0;
  for (int i = 0; i < job.count; ++i) outputs += (double)a.m * job.pr[i].n;
  const double scales = (double)(a.k / a.group_size) * plan.rows_per_block * matrices * (a.symmetric ? 1 : 2);
  // bf16 with a zero point has the longest conversion
  const double expanded = plan.tl * (b4 && a.t_dtype == OFQ_BF16 && !a.symmetric ? 1.2 : 1.0);
  const double reads = tiles * plan.wk * a.m;  // rows of a chunk of x, 256 bytes of them with 4-bit codes
  const double phase = b4 ? 0.075 + 0.53 * expanded + 0.00088 * reads : 0.21 + 0.30 * expanded + 0.00045 * reads;
  return rounds * (5.7 + 0.75 / 4096 * scales + plan.phases * phase) + 1.4e-6 * outputs;
}

// Which of the two streaming kernels takes a job, gemv_rows_mt, whose waves copy x for themselves, or gemv_ring_mt,
// which starts 1.5 us later and takes less per byte.  Both timed on 6065 random jobs of 17 to 64 rows (linears of 512
// to 32000 x 512 to 14336, several of a layer, gated units; weights from HBM): with three tiles of rows a block and
// more gemv_ring_mt takes 0.78 of the time in the mean, 32 of 2290 more than 3 % longer (1.12 at worst, 21 x
// 8380 x 10176 bf16 with a zero point); with one and two tiles 1.21 and 1.02 times, three tiles of 8-bit codes
// with K up to 1024, a phase or two, 1.01 (1037 jobs, 1.19 at worst; from there to 3072 0.95).  (A comparison of
// expected times, with a tenth to spare, turned 824 of the 2310 away: 64 x 11008 x 4096 fp16 4-bit 20.6 us, now 18.6,
// 56 rows 18.7 -> 16.6.)
void gemv_mt_choice(const LinearJob& job, MtChoice* choice) {
  const LinearArgs& a = job.pr[0];
  int64_t total = 0;
  for (int i = 0; i < (job.glu ? 1 : job.count); ++i) total += job.pr[i].n;
  const auto tiles = [&](int64_t rpb) { return (job.glu ? 2 : 1) * ((rpb + 15) / 16); };
  RingMtPlan& plan = choice->plan;
  const int64_t least = job.count == 1 && a.bits == 8 && a.k <= 1024 ? 4 : 3;
  choice->ring = tiles((total + 255) / 256) >= least && ring_mt_plan(job, &plan) && tiles(plan.rows_per_block) >= 3;
  choice->us = choice->ring ? ring_mt_us(job, plan) * 1.05 : rows_mt_us(job);
}
static int launch_mt_job(hipStream_t st, const LinearJob& job, const MtChoice& choice) {
  return choice.ring ? launch_ring_mt(st, job, choice.plan) : launch_rows_mt(st, job);
}

// gemv_flow with 17 to 48 rows of x: expected time in us, within 12 % (17 % with 8-bit codes) of the measured one for 90
// of 100 of 294 random jobs (linears of 512 to 32000 x 512 to 14336, several of a layer, gated units).  A step of the
// longest wave takes a part per KB of x and per KB of codes, which are expanded at a rate of their kind; scales and
// outputs come on top.
static double flow_mt_us(const LinearJob& job, const FlowPlan& plan) {
  const LinearArgs& a = job.pr[0];
  const bool b4 = a.bits == 4;
  const int matrices = job.glu ? 2 : 1;
  const int chunks = flow_chunks(a.bits, plan.mx), ck = b4 ? 128 : 64;
  const int steps = (int)((a.k + chunks * ck - 1) / (chunks * ck));
  double codes = a.symmetric ? 0.226 : 0.230;
  if (b4) codes = a.t_dtype == OFQ_F16 ? (a.symmetric && a.w_signed ? 0.261 : 0.313) : (a.symmetric ? 0.325 : 0.361);
  double outputs = 0;
  for (int i = 0; i < job.count; ++i) outputs += 1e-6 * (double)a.m * job.pr[i].n;
  const double scales = (double)(a.k / a.group_size) * plan.rows_per_block * matrices * (a.symmetric ? 1 : 2) / 4096;
  return (b4 ? 2.7 : 2.4)
         + (steps + plan.nw - 1) / plan.nw
               * ((b4 ? 0.080 : 0.072) * flow_x_ops(a.bits, plan.mx) + codes * chunks * plan.tl * matrices)
         + (b4 ? 0.9 : 1.1) * scales + (b4 ? 6.6 : 7.5) * outputs;
}

// One linear of 17 to 48 rows of x goes to gemv_flow where gemm_wr is not expected to be faster (few rows of a long K:
// 37 x 801 x 13728 17.0 us there, 23.9 here; its second launch as below); several and gated units always do.
// Time over that of the kernels that ran instead (gemv_rows_mt, gemv_ring_mt, gemm_wr), on 330 random jobs with weights
// from HBM: one linear 0.90, with what gemm_wr keeps 0.88, several 0.84 (0.95 at worst), gated units 0.89 (1.02); 24 x
// 11008 x 4096 fp16 4-bit in groups of 32 16.6 -> 13.6 us, 48 x 11008 x 4096 with a zero point 17.2 -> 15.8.  64 rows leave six waves and
// took 1.0 to 1.4 of the time.
bool gemv_flow_preferred(const LinearArgs& a, bool have_workspace, FlowPlan* plan) {
  if (a.m > 48 || !gemv_mt_supported(a)) return false;
  const LinearJob job{&a, 1, false, nullptr, 0};
  if (!flow_plan(job, plan)) return false;
  const double us = flow_mt_us(job, *plan);
  return us < gemm_wr_us(a, have_workspace, us < 12.5 ? 3.0 : 0.5);
}
int launch_flow_tiled(hipStream_t st, const LinearArgs& a, const FlowPlan& plan) {
  return launch_gemv_flow_f16_b4(st, LinearJob{&a, 1, false, nullptr, 0}, plan);
}
int launch_gemv_flow(hipStream_t st, const LinearArgs& a, const FlowPlan& plan) {
  return launch_flow_by(st, LinearJob{&a, 1, false, nullptr, 0}, plan);
}

// gemm_wr reads x once per 128 rows of weights, but starts a second kernel where it slices K: so long
// rows of weights leave the streaming kernels (64 x 4096 x 11008 fp16: 27.6 us here, 17.4 there) and n =
// 11008 of k = 4096 stays.  Below 12.5 us the second launch and the workspace
// have to be won back as well: there the host, 3 us for the two, is what bounds a call that is not replayed
// from a graph.
bool gemv_mt_preferred(const LinearArgs& a, bool have_workspace, MtChoice* choice) {
  if (!gemv_mt_supported(a)) return false;
  gemv_mt_choice(LinearJob{&a, 1, false, nullptr, 0}, choice);
  return choice->us < gemm_wr_us(a, have_workspace, choice->us < 12.5 ? 3.0 : 0.5);
}

int launch_gemv_mt(hipStream_t st, const LinearArgs& a, const MtChoice& choice) {
  return launch_mt_job(st, LinearJob{&a, 1, false, nullptr, 0}, choice);
}

// One launch against one per problem, each by its own best kernel (without a workspace: the entry points of
// several linears and gated units have none), and the gating's: 0.94 of the time at most on 2429 random layers, 0.53 in
// the mean, with gemv_ring_mt where it takes them.  gemv_rows_mt on three tiles a block and more (rows of K whose
// scales leave gemv_ring_mt no room) by expected times.
int launch_gemv_mt_several(hipStream_t st, const LinearArgs* pr, int count, bool glu, void* y, int act) {
  if (count < 2 || count > kGemvMaxProblems) return OFQ_ERR_UNSUPPORTED;
  const LinearArgs& a = pr[0];
  for (int i = 0; i < count; ++i) {
    const LinearArgs& b = pr[i];
    if (!gemv_mt_supported(b) || b.t_dtype != a.t_dtype || b.bits != a.bits || b.w_signed != a.w_signed
        || b.symmetric != a.symmetric || b.group_size != a.group_size || b.m != a.m || b.k != a.k
        || (glu && (b.x != a.x || b.n != a.n))) {
      return OFQ_ERR_UNSUPPORTED;
    }
  }
  const LinearJob job{pr, count, glu, y, act};
  FlowPlan flow;
  if (a.m <= 48 && flow_plan(job, &flow)) return launch_flow_by(st, job, flow);
  MtChoice choice;
  gemv_mt_choice(job, &choice);
  if (!choice.ring) {
    double apart = glu ? 4.0 : 0.0;
    for (int i = 0; i < count; ++i) {
      MtChoice one;
      gemv_mt_choice(LinearJob{&pr[i], 1, false, nullptr, 0}, &one);
      const double wr = gemm_wr_us(pr[i], false, 0.0);
      apart += one.us < wr ? one.us : wr;
    }
    if (choice.us > apart) return OFQ_ERR_UNSUPPORTED;
  }
  return launch_mt_job(st, job, choice);
}

bool gemv_wq_supported(const LinearArgs& a) {
  if (rows_supported(a)) return true;
  if (a.t_dtype != OFQ_F16 || a.group_dim != 1 || a.m > 16 || a.m < 1) return false;
  const int ch = a.bits == 4 ? 128 : 64;
  const int lk = ch / 4;
  if (a.k % ch != 0 || a.group_size % lk != 0) return false;
  if (a.n * a.k > 0x7FFFFFFFLL * 8 || a.k > 0x7FFFFFFF || a.n > 0x7FFFFFFF - 16) return false;
  return true;
}

int launch_gemv_wq(hipStream_t st, const LinearArgs& a) {
  if (gemv_m1_supported(a)) {
    const int rc = launch_gemv_m1(st, a);
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  if (gemv_m1_any_supported(a)) {
    const int rc = launch_gemv_m1_any(st, a);
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  {
    const int rc = launch_flow(st, LinearJob{&a, 1, false, nullptr, 0});
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  if (w4s_supported(a)) {
    const int rc = launch_w4s(st, a);
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  } else if (w4p_supported(a)) {
    // uint8 container / asymmetric: the row-balanced kernel with the reference's roundings
    const int rc = launch_w4p(st, a, ilog2_exact(a.group_size / 128), false);
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  if (rows_supported(a)) {
    const int rc = launch_rows(st, a);
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  if (a.t_dtype != OFQ_F16) return OFQ_ERR_UNSUPPORTED;  // the kernels below are fp16 only
  {
    const int ch = a.bits == 4 ? 128 : 64;
    if (a.k % ch != 0 || a.group_size % (ch / 4) != 0) return OFQ_ERR_UNSUPPORTED;
  }
  const int zmode = !a.symmetric ? kZeroAsym : (a.w_signed ? kZeroNone : kZeroSymU);
#define OFQ_V(B, SG, ZM) \
  if (a.bits == B && a.w_signed == SG && zmode == ZM) return launch_gemv_variant<B, SG, ZM>(st, a);
  OFQ_V(4, true, kZeroNone)
  OFQ_V(4, false, kZeroSymU)
  OFQ_V(4, false, kZeroAsym)
  OFQ_V(8, true, kZeroNone)
  OFQ_V(8, false, kZeroSymU)
  OFQ_V(8, false, kZeroAsym)
#undef OFQ_V
  return OFQ_ERR_UNSUPPORTED;
}

int launch_linear_generic(hipStream_t st, const LinearArgs& a) {
  if (rows_f32_supported(a)) {
    const int rc = launch_rows_f32(st, a);
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;
  }
  if (a.m > 65535) return OFQ_ERR_UNSUPPORTED;
  switch (a.t_dtype) {
    case OFQ_F16: return launch_generic_t<f16>(st, a);
    case OFQ_BF16: return launch_generic_t<bf16>(st, a);
    case OFQ_F32: return launch_generic_t<float>(st, a);
    default: return OFQ_ERR_BAD_DTYPE;
  }
}

}  // namespace ofq

using namespace ofq;

extern "C" size_t ofq_fused_linear_gq_workspace_bytes(int w_dtype, int t_dtype, int num_bits,
                                                      int symmetric, int group_dim,
                                                      int64_t group_size, int64_t m, int64_t n,
                                                      int64_t k) {
  if ((num_bits != 4 && num_bits != 8) || group_size <= 0 || m <= 0 || n <= 0 || k <= 0) return 0;
  LinearArgs a{};
  a.t_dtype = t_dtype;
  a.w_signed = w_dtype == OFQ_I8;
  a.bits = num_bits;
  a.symmetric = symmetric != 0;
  a.group_dim = group_dim;
  a.group_size = group_size;
  a.m = m;
  a.n = n;
  a.k = k;
  MtChoice choice;
  if (gemv_wq_supported(a) || gemv_m1_any_supported(a) || gemv_mt_preferred(a, true, &choice)) return 0;
  if (group_dim == 0) return gemm_gn_workspace_bytes(a);
  return gemm_wq_workspace_bytes(a);  // K slices, from 1024 rows on at least the converted weight
}

extern "C" int ofq_fused_linear_gq(void* stream, const void* x, const void* w,
                                   const void* w_scale, const void* w_zero, const void* b,
                                   void* out, int w_dtype, int t_dtype, int num_bits,
                                   int symmetric, int group_dim, int64_t group_size, int64_t m,
                                   int64_t n, int64_t k, void* workspace, size_t workspace_bytes) {
  // checks of FusedLinearWithGroupwiseQuantizedWeightKernel::Compute,
  // groupwise_quantization_kernels.cu:773-822
  OFQ_RETURN_IF(num_bits != 4 && num_bits != 8, OFQ_ERR_BAD_ATTR);
  OFQ_RETURN_IF(group_dim != 0 && group_dim != 1, OFQ_ERR_BAD_ATTR);
  OFQ_RETURN_IF(w_dtype != OFQ_U8 && w_dtype != OFQ_I8, OFQ_ERR_BAD_DTYPE);
  OFQ_RETURN_IF(!symmetric && w_dtype != OFQ_U8, OFQ_ERR_BAD_DTYPE);
  OFQ_RETURN_IF(t_dtype != OFQ_F16 && t_dtype != OFQ_BF16 && t_dtype != OFQ_F32,
                OFQ_ERR_BAD_DTYPE);
  OFQ_RETURN_IF(m < 0 || n < 0 || k <= 0, OFQ_ERR_BAD_SHAPE);
  OFQ_RETURN_IF(k % (8 / num_bits) != 0, OFQ_ERR_BAD_SHAPE);
  const int64_t group_dim_size = group_dim == 0 ? n : k;
  OFQ_RETURN_IF(group_size <= 0, OFQ_ERR_BAD_ATTR);
  if (m == 0 || n == 0) return OFQ_OK;
  OFQ_RETURN_IF(group_size > group_dim_size || group_dim_size % group_size != 0,
                OFQ_ERR_BAD_SHAPE);
  // int32 index limits of the reference launchers, :651-655
  const int64_t i32max = 0x7FFFFFFF;
  OFQ_RETURN_IF(m * k > i32max || n * k > i32max || m * n > i32max, OFQ_ERR_UNSUPPORTED);
  OFQ_RETURN_IF(x == nullptr || w == nullptr || w_scale == nullptr || out == nullptr,
                OFQ_ERR_NULL_POINTER);
  OFQ_RETURN_IF((symmetric != 0) != (w_zero == nullptr), OFQ_ERR_NULL_POINTER);
  OFQ_RETURN_IF(!ofq_aligned16(x) || !ofq_aligned16(w) || !ofq_aligned16(w_scale)
                    || !ofq_aligned16(w_zero) || !ofq_aligned16(b) || !ofq_aligned16(out),
                OFQ_ERR_MISALIGNED);
  LinearArgs a;
  a.x = x;
  a.w = w;
  a.scale = w_scale;
  a.zero = w_zero;
  a.bias = b;
  a.out = out;
  a.t_dtype = t_dtype;
  a.w_signed = w_dtype == OFQ_I8;
  a.bits = num_bits;
  a.symmetric = symmetric != 0;
  a.group_dim = group_dim;
  a.group_size = group_size;
  a.m = m;
  a.n = n;
  a.k = k;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // (the row-per-wave kernel for one row of x covers rows and groups off the chunk grid of the
  // MFMA kernels: k a multiple of 32 / 16 elements, groups from 32 / 16)
  if (gemv_wq_supported(a) || gemv_m1_any_supported(a)) {
    const int rc = launch_gemv_wq(st, a);
    if (rc != OFQ_ERR_UNSUPPORTED) return rc;  // e.g. bf16 with an x too large to stage
  }
  if (a.m > 16 && a.m <= 64) {
    const bool have_workspace = workspace != nullptr && workspace_bytes >= gemm_wq_workspace_bytes(a);
    FlowPlan flow;
    if (gemv_flow_preferred(a, have_workspace, &flow)) return launch_gemv_flow(st, a, flow);
    MtChoice choice;
    if (gemv_mt_preferred(a, have_workspace, &choice)) {
      const int rc = launch_gemv_mt(st, a, choice);
      if (rc != OFQ_ERR_UNSUPPORTED) return rc;
    }
  }
  if (gemm_wq_supported(a)) return launch_gemm_wq(st, a, workspace, workspace_bytes);
  if (a.group_dim == 0) {
    const size_t need = gemm_gn_workspace_bytes(a);
    if (need != 0 && workspace != nullptr && workspace_bytes >= need && ofq_aligned16(workspace)) {
      return launch_gemm_gn(st, a, workspace);
    }
    if (gemv_gn_supported(a)) {
      const int rc = launch_gemv_gn(st, a);
      if (rc != OFQ_ERR_UNSUPPORTED) return rc;
    }
  }
  return launch_linear_generic(st, a);
}

// ---- tile-major weight copy -------------------------------------------------------------------
namespace ofq {
namespace {

// one lane moves the 16 bytes it will later request: lane (k-slot kb, row r) of chunk c of tile t
// of block b <- row b * rows_per_block + 16 t + r, bytes [64 c + 16 kb, +16); rows past the
// block's share (or past n) become zeros
__global__ void __launch_bounds__(256)
repack_w4_tiles(const uint8_t* __restrict__ w, uint8_t* __restrict__ tiled, int N, int K,
                int rows_per_block, int tiles_per_block, int64_t pieces) {
  const int nchunks = K >> 7;
  const int row_bytes = K >> 1;
  for (int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x; p < pieces;
       p += (int64_t)gridDim.x * 256) {
    const int lane = (int)(p & 63);
    const int64_t kb_index = p >> 6;  // (block * tiles_per_block + t) * nchunks + c
    const int c = (int)(kb_index % nchunks);
    const int64_t tile_index = kb_index / nchunks;
    const int t = (int)(tile_index % tiles_per_block);
    const int64_t b = tile_index / tiles_per_block;
    const int r = lane & 15, kb = lane >> 4;
    const int row_l = 16 * t + r;
    const int64_t row = b * rows_per_block + row_l;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (row_l < rows_per_block && row < N) {
      v = *reinterpret_cast<const u32x4*>(w + row * row_bytes + c * 64 + kb * 16);
    }
    reinterpret_cast<u32x4*>(tiled)[p] = v;
  }
}

bool tiled_shape_ok(int num_bits, int64_t n, int64_t k) {
  return num_bits == 4 && n >= 1 && k >= 128 && k % 128 == 0 && k <= (1 << 20)
         && n <= 0x7FFFFFFF - 16;
}

}  // namespace
}  // namespace ofq

extern "C" size_t ofq_groupwise_repack_bytes(int num_bits, int64_t n, int64_t k) {
  if (!tiled_shape_ok(num_bits, n, k)) return 0;
  int64_t grid;
  int rpb;
  w4p_row_split(n, &grid, &rpb);
  return (size_t)grid * (size_t)((rpb + 15) / 16) * 16 * (size_t)(k / 2);
}

extern "C" int ofq_groupwise_repack(void* stream, const void* w, void* w_tiled, int num_bits,
                                    int64_t n, int64_t k) {
  OFQ_RETURN_IF(num_bits != 4 && num_bits != 8, OFQ_ERR_BAD_ATTR);
  OFQ_RETURN_IF(n <= 0 || k <= 0, OFQ_ERR_BAD_SHAPE);
  OFQ_RETURN_IF(!tiled_shape_ok(num_bits, n, k), OFQ_ERR_UNSUPPORTED);
  OFQ_RETURN_IF(w == nullptr || w_tiled == nullptr, OFQ_ERR_NULL_POINTER);
  OFQ_RETURN_IF(!ofq_aligned16(w) || !ofq_aligned16(w_tiled), OFQ_ERR_MISALIGNED);
  int64_t grid;
  int rpb;
  w4p_row_split(n, &grid, &rpb);
  const int tpb = (rpb + 15) / 16;
  const int64_t pieces = grid * tpb * (k / 128) * 64;
  int64_t blocks = (pieces + 255) / 256;
  if (blocks > 256 * 64) blocks = 256 * 64;
  repack_w4_tiles<<<(unsigned)blocks, 256, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const uint8_t*>(w), static_cast<uint8_t*>(w_tiled), (int)n, (int)k, rpb, tpb,
      pieces);
  return ofq_check_launch();
}

extern "C" int ofq_fused_linear_gq_tiled(void* stream, const void* x, const void* w_tiled,
                                         const void* w_scale, const void* w_zero, const void* b,
                                         void* out, int w_dtype, int t_dtype, int num_bits,
                                         int symmetric, int group_dim, int64_t group_size,
                                         int64_t m, int64_t n, int64_t k) {
  OFQ_RETURN_IF(num_bits != 4 && num_bits != 8, OFQ_ERR_BAD_ATTR);
  OFQ_RETURN_IF(group_dim != 0 && group_dim != 1, OFQ_ERR_BAD_ATTR);
  OFQ_RETURN_IF(w_dtype != OFQ_U8 && w_dtype != OFQ_I8, OFQ_ERR_BAD_DTYPE);
  OFQ_RETURN_IF(!symmetric && w_dtype != OFQ_U8, OFQ_ERR_BAD_DTYPE);
  OFQ_RETURN_IF(t_dtype != OFQ_F16 && t_dtype != OFQ_BF16 && t_dtype != OFQ_F32,
                OFQ_ERR_BAD_DTYPE);
  OFQ_RETURN_IF(m < 0 || n < 0 || k <= 0 || group_size <= 0, OFQ_ERR_BAD_SHAPE);
  if (m == 0 || n == 0) return OFQ_OK;
  const int64_t group_dim_size = group_dim == 0 ? n : k;
  OFQ_RETURN_IF(group_size > group_dim_size || group_dim_size % group_size != 0,
                OFQ_ERR_BAD_SHAPE);
  OFQ_RETURN_IF(x == nullptr || w_tiled == nullptr || w_scale == nullptr || out == nullptr,
                OFQ_ERR_NULL_POINTER);
  OFQ_RETURN_IF((symmetric != 0) != (w_zero == nullptr), OFQ_ERR_NULL_POINTER);
  OFQ_RETURN_IF(!ofq_aligned16(x) || !ofq_aligned16(w_tiled) || !ofq_aligned16(w_scale)
                    || !ofq_aligned16(w_zero) || !ofq_aligned16(b) || !ofq_aligned16(out),
                OFQ_ERR_MISALIGNED);
  LinearArgs a;
  a.x = x;
  a.w = w_tiled;
  a.scale = w_scale;
  a.zero = w_zero;
  a.bias = b;
  a.out = out;
  a.t_dtype = t_dtype;
  a.w_signed = w_dtype == OFQ_I8;
  a.bits = num_bits;
  a.symmetric = symmetric != 0;
  a.group_dim = group_dim;
  a.group_size = group_size;
  a.m = m;
  a.n = n;
  a.k = k;
  // what the row-balanced kernel takes: fp16, 4 bits, groups of a multiple of 128 along K, at
  // most 16 rows of x whose m * k halves fit LDS
  if (!w4p_supported(a) || !tiled_shape_ok(num_bits, n, k)) return OFQ_ERR_UNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
  FlowPlan flow;
  if (a.m > 1 && gemv_flow_choice(LinearJob{&a, 1, false, nullptr, 0}, &flow)) {
    flow.tiled = 1;
    return launch_flow_tiled(st, a, flow);
  }
  return launch_w4p(st, a, ilog2_exact(a.group_size / 128), true);
}
