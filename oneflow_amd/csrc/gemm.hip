// MFMA GEMMs for gfx950:
//   (1) fused_linear_with_groupwise_quantized_weight for m > 16: either the weight tile is
//       dequantised on its way into LDS and feeds fp16/bf16 MFMA (the fp16/bf16 copy of the
//       weight that the reference materialises for m > 8,
//       oneflow/core/functional/impl/quantization.cpp:341-350, then never touches HBM), cut
//       along K into separate blocks when a workspace for partial sums is given and the tiles
//       alone would not fill the chip; or, at large m with a workspace, the weight is
//       dequantised once and a copy-fed GEMM runs on it;
//   (2) matmul_quant: int8 x int8 -> int32 MFMA with a per-row/per-tensor scale epilogue.
//
// Three kernels share one layout: a tile row is always 128 bytes of K (64 fp16/bf16 or 128 int8
// elements), a k-step of the 32x32 MFMA consumes 32 of those bytes per row (16 bytes per lane), whatever
// the type.  gemm_core2 (gemm_kernels.h) serves both operations, gemm_pp (gemm_pp.h) their copy-fed
// tiles of 256 rows, gemm_wr (gemm_wr.h) 17 rows and more with the weights packed up to the registers.
// This file only chooses kernel, tile and slices and fills parameter blocks.
#include <cmath>

#include "gemm_deep.h"
#include "gemm_kernels.h"
#include "ofq_device.h"
#include "ofq_internal.h"

namespace ofq {

// Width of the weight tile under a 256-row tile of x in the in-tile path.  The blocks run in rounds of one per
// CU; a round costs about in proportion to the tile width, so the one with the smaller (rounds x width) wins,
// the wider one on a tie (less L2 -> LDS traffic per MFMA): 192 turns the 258 or 344 tiles of m = 768 /
// 1024 at n = 11008 (two rounds of 128-wide tiles, the second nearly empty) into one round of 174 / 232:
// 160 -> 115 us.
int pick_tile_width(int64_t m, int64_t n) {
  const int64_t m_tiles = (m + 255) / 256;
  auto cost = [&](int64_t bn) { return ((m_tiles * ((n + bn - 1) / bn) + 255) / 256) * bn; };
  return cost(192) <= cost(128) ? 192 : 128;
}

namespace {

inline int ceil_div(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }

// The GEMMs whose operands are both copied (int8, and 16-bit behind a converted weight): their tiles, and the
// expected time in us of one on m x n outputs and kt k-tiles of 128 bytes,
//   start + outputs * m n / 10^6 + kt * (alone + share * b/256 + round * ceil(b/256) + pair * ceil(b/512)
//                                        + four * ceil(b/1024))
// with b blocks: tiles from 256 rows on run one block a CU (rounds of 256), those of 128 two, those of 64 four (of
// int8's, kCopyCostI8, as many as their stages leave room for).
// 16 bits: fitted to 384 random problems of 1024 to 4096 rows, to 32000 columns and k to 14336; on 2900 others
// 0.74 of what the rules chose, 14 more than 3 % longer (1.14 at worst, 1609 x 12072 x 576, where 384 columns are
// the best tile and 192 the chosen one).
enum CopyTile { kCopy64, kCopy128, kCopy256x128, kCopy256x192, kCopy256x256, kCopy256x384, kCopyTiles };
struct TileCost {
  int bm, bn;
  double start, outputs, alone, share, round, pair, four;
};
const TileCost kCopyCost[2][kCopyTiles] = {  // [ragged k]
    {{64, 64, 5.1, 0.17, 0.088, 0.194, 0.038, 0.0, 0.0},
     {128, 128, 4.3, 0.73, 0.0, 0.189, 0.013, 0.534, 0.0},
     {256, 128, 5.8, 0.71, 0.0, 0.203, 0.778, 0.0, 0.0},
     {256, 192, 8.6, 0.70, 0.0, 0.303, 0.887, 0.0, 0.0},
     {256, 256, 10.6, 0.75, 0.0, 0.469, 0.952, 0.0, 0.0},
     {256, 384, 13.9, 0.66, 0.0, 0.617, 1.324, 0.0, 0.0}},
    {{64, 64, 4.5, 0.37, 0.139, 0.151, 0.115, 0.0, 0.0},
     {128, 128, 4.4, 0.47, 0.0, 0.174, 0.204, 0.466, 0.0},
     {256, 128, 4.1, 0.84, 0.0, 0.027, 1.042, 0.0, 0.0},
     {256, 192, 8.0, 0.54, 0.0, 0.316, 1.100, 0.0, 0.0},
     {256, 256, 9.9, 0.66, 0.0, 0.382, 1.310, 0.0, 0.0},
     {256, 384, 14.6, 0.54, 0.0, 0.586, 1.697, 0.0, 0.0}}};
// int8: fitted to 9158 random products of 65 to 8192 rows, 512 to 14336 columns and k from 512 to 8192, a third of them
// with a ragged last k-tile, each timed on every tile with weights from HBM: within 10 to 16 % of the measured time for
// 90 of 100.  The choice (with the slices of mq_plan and the streaming kernel) takes 1.2 % longer than the best one in
// the mean.  Of the tiles of gemm_deep the ones of fewer stages leave room for a second and third block, whose
// products lie under the first one's epilogue: they win where K is short and blocks are many; 128 x 128 does
// so with two stages of gemm_core2 (1852 x 8323 x 512 19.2 us there, 26.3 with five stages).
// Time over that of one k-tile under way on every tile (gemm_core2, its own fitted choice, with its slices): 0.72 in the mean at 65 to
// 128 rows, 0.80 to 256, 0.81 to 512, 0.85 to 1024, 0.88 to 2048, 0.95 to 8192; 256 x 4096 x 4096 26.5 -> 13.0 us,
// 512 x 4096 x 4096 27.7 -> 17.2, 1024 x 4096 x 4096 33.4 -> 25; 5 of 100 take more than 3 % longer, to 1.35 (rows of
// 512 elements, 190 x 775 x 2496 10.4 -> 14.0).
enum MqTile {
  kMq64, kMq64Short, kMq128x64, kMq128x64Short, kMq128, kMq128Short, kMq256x128, kMq256x192, kMq256x256, kMq256x384,
  kMqTiles
};
const TileCost kCopyCostI8[2][kMqTiles] = {  // [ragged k]
    {{64, 64, 3.29, 1.088, 0.0, 0.005, 0.187, 0.107, 0.0},
     {64, 64, 3.22, 0.516, 0.0, 0.121, 0.049, 0.085, 0.136},
     {128, 64, 3.46, 1.442, 0.0, 0.076, 0.315, 0.0, 0.0},
     {128, 64, 3.27, 0.607, 0.0, 0.166, 0.123, 0.187, 0.0},
     {128, 128, 4.49, 1.016, 0.0, 0.117, 0.449, 0.0, 0.0},
     {128, 128, 3.36, 0.681, 0.0, 0.214, 0.0, 0.684, 0.0},
     {256, 128, 6.46, 0.754, 0.0, 0.183, 0.649, 0.0, 0.0},
     {256, 192, 8.86, 0.515, 0.0, 0.314, 1.039, 0.0, 0.0},
     {256, 256, 10.39, 0.485, 0.0, 0.305, 1.247, 0.0, 0.0},
     {256, 384, 14.53, 0.423, 0.0, 0.528, 1.506, 0.0, 0.0}},
    {{64, 64, 3.19, 1.057, 0.0, 0.004, 0.183, 0.244, 0.0},
     {64, 64, 3.10, 0.681, 0.0, 0.040, 0.114, 0.131, 0.200},
     {128, 64, 3.36, 1.477, 0.0, 0.038, 0.457, 0.0, 0.0},
     {128, 64, 3.26, 0.630, 0.0, 0.068, 0.257, 0.204, 0.0},
     {128, 128, 4.19, 1.048, 0.0, 0.050, 0.610, 0.0, 0.0},
     {128, 128, 3.19, 0.662, 0.0, 0.213, 0.073, 0.703, 0.0},
     {256, 128, 6.16, 0.755, 0.0, 0.088, 0.897, 0.0, 0.0},
     {256, 192, 8.54, 0.422, 0.0, 0.286, 1.299, 0.0, 0.0},
     {256, 256, 10.32, 0.461, 0.0, 0.253, 1.631, 0.0, 0.0},
     {256, 384, 14.67, 0.488, 0.0, 0.349, 1.973, 0.0, 0.0}}};

double tile_us(const TileCost& c, int64_t m, int64_t n, int64_t kt, int splits = 1) {
  const double b = (double)((m + c.bm - 1) / c.bm) * (double)((n + c.bn - 1) / c.bn) * splits;
  return c.start + c.outputs * 1e-6 * (double)m * n
         + kt * (c.alone + c.share * b / 256 + c.round * std::ceil(b / 256) + c.pair * std::ceil(b / 512)
                 + c.four * std::ceil(b / 1024));
}
int pick_tile(const TileCost* cost, int tiles, int64_t m, int64_t n, int64_t row_bytes, double* us) {
  int best = 0;
  double best_us = 1e300;
  for (int i = 0; i < tiles; ++i) {
    const double t = tile_us(cost[i], m, n, (row_bytes + 127) / 128);
    if (t < best_us) {
      best = i;
      best_us = t;
    }
  }
  *us = best_us;
  return best;
}
CopyTile pick_copy_tile(int64_t m, int64_t n, int64_t row_bytes, double* us) {
  return (CopyTile)pick_tile(kCopyCost[row_bytes % 128 != 0], kCopyTiles, m, n, row_bytes, us);
}

}  // namespace

namespace {

// x[m,k] * wt[n,k]^T with both operands in T (the dequantised weight of the two-pass path)
template<bool RG, typename T, class MF>
int launch_plain(hipStream_t st, const LinearArgs& a, const void* wt) {
  typedef typename TT<T>::storage S;
  typedef EpBias<T> EP;
  BCopyParams bp;
  bp.b = static_cast<const uint8_t*>(wt);
  bp.ldb = a.k * 2;
  bp.N = (int)a.n;
  typename EP::Params ep;
  ep.bias = static_cast<const S*>(a.bias);
  ep.out = static_cast<S*>(a.out);
  const int64_t kt = (a.k + 63) / 64;
  double us;
  const CopyTile tile = pick_copy_tile(a.m, a.n, a.k * 2, &us);
  switch (tile) {
    case kCopy64:
      return launch_core2<MF, B2Copy<RG, 64, 256>, EP, 64, 64, 2, 2>(st, a.x, a.k * 2, bp, ep, a.m, a.n, kt);
    case kCopy128:
      return launch_core2<MF, B2Copy<RG, 128, 512>, EP, 128, 128, 4, 2>(st, a.x, a.k * 2, bp, ep, a.m, a.n, kt);
    case kCopy256x128:
      return launch_core2<MF, B2Copy<RG, 128, 512>, EP, 256, 128, 4, 2>(st, a.x, a.k * 2, bp, ep, a.m, a.n, kt);
    default: break;
  }
  if constexpr (RG) {  // (why: launch_pp)
    if (tile == kCopy256x192) {
      return launch_core2<MF, B2Copy<RG, 192, 512>, EP, 256, 192, 4, 2>(st, a.x, a.k * 2, bp, ep, a.m, a.n, kt);
    }
    if (tile == kCopy256x256) {
      return launch_core2<MF, B2Copy<RG, 256, 512>, EP, 256, 256, 4, 2>(st, a.x, a.k * 2, bp, ep, a.m, a.n, kt);
    }
  }
  const int width = kCopyCost[RG][tile].bn;
  return std::is_same<T, f16>::value
             ? launch_gemm_pp_f16(st, a.x, wt, a.bias, a.out, a.m, a.n, a.k, width)
             : launch_gemm_pp_bf16(st, a.x, wt, a.bias, a.out, a.m, a.n, a.k, width);
}

// Few blocks (m small against the tile height, or few weight tiles): K is cut into `splits`
// slices that run as separate blocks, each writing fp32 partial sums of the whole output tile to
// its slice of the workspace; splitk_finalize adds the slices in order (so the result does not
// depend on scheduling), adds the bias and rounds to T once.
//
// Four outputs a thread at a flat index of [M, N], the last thread's four end with the last output (M N >= 4;
// what two threads compute is the same).  Rows of N and slices of M N elements begin at any element.
template<typename V, typename E>
__device__ __forceinline__ V sum_slices4(const E* __restrict__ part, int64_t MN, int splits) {
  typedef V any __attribute__((aligned(4)));
  constexpr int U = 4;  // slices requested together
  V sum = *reinterpret_cast<const any*>(part);
  for (int s0 = 1; s0 < splits; s0 += U) {
    V v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      v[u] = *reinterpret_cast<const any*>(part + (int64_t)(s0 + u < splits ? s0 + u : splits - 1) * MN);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s0 + u < splits) sum += v[u];
  }
  return sum;
}
template<typename T, typename F>
__device__ __forceinline__ void store_folded4(typename TT<T>::storage* __restrict__ out, int n, int N,
                                              F value) {
  typename TT<T>::storage o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    TT<T>::store(&o[e], value(e, n));
    if (++n == N) n = 0;
  }
  if constexpr (sizeof(o) == 8) {
    *reinterpret_cast<u32x2_any*>(out) = *reinterpret_cast<const u32x2*>(o);
  } else {
    *reinterpret_cast<u32x4_any*>(out) = *reinterpret_cast<const u32x4*>(o);
  }
}

template<typename T>
__global__ void __launch_bounds__(256)
splitk_finalize(const float* __restrict__ part, const typename TT<T>::storage* __restrict__ bias,
                typename TT<T>::storage* __restrict__ out, uint32_t MN, uint32_t N, int splits) {
  uint32_t i = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= MN) return;
  i = i < MN - 4 ? i : MN - 4;
  const f32x4 acc = sum_slices4<f32x4>(part + i, MN, splits);
  store_folded4<T>(out + i, (int)(i % N), (int)N, [&](int e, int n) {
    return bias != nullptr ? acc[e] + TT<T>::load(bias + n) : acc[e];
  });
}

// Slices of K for the in-tile path: as many as still fit the blocks into one resident round
// (256x128 tiles: one 8-wave block per CU; 128x128: two 4-wave blocks), each at least 4 k-tiles.
int wq_splits(const LinearArgs& a) {
  if (a.m >= 1024) return 1;  // two-pass territory
  const int64_t bm = a.m > 128 ? 256 : 128;
  const int64_t slots = a.m > 128 ? 256 : 512;
  const int64_t blocks = ((a.m + bm - 1) / bm) * ((a.n + 127) / 128);
  int64_t s = slots / blocks;
  const int64_t kt = (a.k + 63) / 64;
  if (s > 8) s = 8;
  if (s > kt / 4) s = kt / 4;
  if (s < 1) s = 1;
  // no empty last slice
  while (s > 1 && ((kt + s - 1) / s) * (s - 1) >= kt) --s;
  return (int)s;
}

template<bool RG, typename T, class MF, int BITS, bool SIGNED, int ZMODE>
int launch_wq_variant(hipStream_t st, const LinearArgs& a, float* partials, int splits) {
  typedef typename TT<T>::storage S;
  typedef EpBias<T> EP;
  WqParams<T> bp;
  bp.w = static_cast<const uint8_t*>(a.w);
  bp.scale = static_cast<const S*>(a.scale);
  bp.zero = static_cast<const S*>(a.zero);
  bp.ldw = a.k * BITS / 8;
  bp.N = (int)a.n;
  bp.G = (int)(a.k / a.group_size);
  bp.group_size = (int)a.group_size;
  typename EP::Params ep;
  ep.bias = static_cast<const S*>(a.bias);
  ep.out = static_cast<S*>(a.out);
  if (partials != nullptr && splits > 1) {
    EpPartial::Params pp;
    pp.out = partials;
    int rc;
    if (a.m > 128) {
      rc = launch_core2<MF, B2Dequant<RG, T, BITS, SIGNED, ZMODE, 128, 512>, EpPartial, 256, 128, 4,
                        2>(st, a.x, a.k * 2, bp, pp, a.m, a.n, (a.k + 63) / 64, splits);
    } else {
      // 8 waves on the 128x128 tile (32x64 per wave): more waves to hide the slice's short
      // k loop behind (28 us against 33 us on 4 waves at m = 128, 11008x4096)
      rc = launch_core2<MF, B2Dequant<RG, T, BITS, SIGNED, ZMODE, 128, 512>, EpPartial, 128, 128, 4,
                        2>(st, a.x, a.k * 2, bp, pp, a.m, a.n, (a.k + 63) / 64, splits);
    }
    if (rc != OFQ_OK) return rc;
    const int64_t mn = a.m * a.n;
    splitk_finalize<T><<<(unsigned)((mn + 1023) / 1024), 256, 0, st>>>(
        partials, ep.bias, ep.out, (uint32_t)mn, (uint32_t)a.n, splits);
    return ofq_check_launch();
  }
  // 256x128 tiles on 8 waves when there are enough rows of x to fill them, else 128x128 on 4
  if (a.m > 128) {
    if (pick_tile_width(a.m, a.n) == 192) {
      return launch_core2<MF, B2Dequant<RG, T, BITS, SIGNED, ZMODE, 192, 512>, EP, 256, 192, 4, 2>(
          st, a.x, a.k * 2, bp, ep, a.m, a.n, (a.k + 63) / 64);
    }
    return launch_core2<MF, B2Dequant<RG, T, BITS, SIGNED, ZMODE, 128, 512>, EP, 256, 128, 4, 2>(
        st, a.x, a.k * 2, bp, ep, a.m, a.n, (a.k + 63) / 64);
  }
  // few rows of x: 128-wide weight tiles would leave most CUs without a block (86 tiles for
  // n = 11008), so the weight tile shrinks until the grid covers the chip
  const int64_t n_tiles128 = (a.n + 127) / 128;
  if (n_tiles128 < 192) {
    return launch_core2<MF, B2Dequant<RG, T, BITS, SIGNED, ZMODE, 32, 256>, EP, 128, 32, 4, 1>(
        st, a.x, a.k * 2, bp, ep, a.m, a.n, (a.k + 63) / 64);
  }
  return launch_core2<MF, B2Dequant<RG, T, BITS, SIGNED, ZMODE, 128, 256>, EP, 128, 128, 2, 2>(
      st, a.x, a.k * 2, bp, ep, a.m, a.n, (a.k + 63) / 64);
}

template<typename T, class MF>
int launch_wq_t(hipStream_t st, const LinearArgs& a, float* partials, int splits) {
  const int zmode = !a.symmetric ? 2 : (a.w_signed ? 0 : 1);
#define OFQ_V(B, SG, ZM)                                                                       \
  if (a.bits == B && a.w_signed == SG && zmode == ZM)                                          \
    return a.k % 64 == 0 ? launch_wq_variant<false, T, MF, B, SG, ZM>(st, a, partials, splits) \
                         : launch_wq_variant<true, T, MF, B, SG, ZM>(st, a, partials, splits);
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

bool gemm_wq_supported(const LinearArgs& a) {
  if (a.t_dtype != OFQ_F16 && a.t_dtype != OFQ_BF16) return false;
  if (a.group_dim != 1 || a.m < 1) return false;
  const int elems_per_chunk = a.bits == 4 ? 32 : 16;
  // whole chunks of codes (and whole 16-byte pieces of x) per row; a last k-tile that is not full
  // is padded with zeros in LDS
  if (a.k % elems_per_chunk != 0 || a.group_size % elems_per_chunk != 0) return false;
  return true;
}

namespace {

// Expected times in us, fitted to 84 000 timings (n from 512 to 32000, half of them odd, k from 512 to 14336,
// 17 <= m <= 1020, both types, both widths, with and without a zero point, groups of 32, 64 and 128, weights
// not in cache).  They are within 18 % of the measured time for 98 of 100 plans; the plan chosen takes
// 1.5 % longer than the fastest one in the mean (3 % at 65 to 128 rows).
//
// `blocks` blocks on `slots` places: a k-step costs `alone` us where a block has the chip to itself and
// `full` where every place is taken (the copies share the L2s, the matrix cores a clock).
double rounds_us(int blocks, int slots, double alone, double full) {
  const int rest = blocks % slots;
  return blocks / slots * full + (rest != 0 ? alone + (full - alone) * rest / slots : 0.0);
}

inline bool has_zero_term(const LinearArgs& a) { return !a.symmetric || !a.w_signed; }

// Tile and K slices of gemm_wr for more than 16 rows (fewer stream) by the least expected time:
//   the start, and 1.9 per 4096 scales (and zeros) that a block copies first;
//   the steps, measured with symmetric fp16 4-bit codes; others take longer to expand, which the taller
//   tiles hide better; a K that is not whole steps costs 1.4 times as much (the copies of such a
//   kernel are all waited for); 8-bit codes that a single block reads are bound by the stream of them;
//   the end: the output, whose rows begin anywhere in a line where n is not whole pieces of 16 bytes, or for
//   slices the second launch and their fp32 sums out and back at 5.2 TB/s.
// Without a workspace the sums of slices have nowhere to go: the tile that is best with one slice.
double wr_plan_us(const LinearArgs& a, bool have_workspace, WrPlan* plan) {
  double best = 1e30;
  if (a.m <= 16) return best;
  if (a.group_size % 32 != 0 || a.k % 32 != 0) return best;
  // k / group_size as a multiply-high by ceil(2^32 / group_size) is exact up to here
  if ((a.group_size & (a.group_size - 1)) != 0 && a.k * a.group_size >= ((int64_t)1 << 32)) return best;
  struct Tile {
    WrTile tile;
    int bm, bn, step_k;
    int above;  // up to so many rows the tile before does the same in less time
    double start, alone, full;
    bool any_bits, tall;
  };
  static const Tile tiles[] = {{kWr32x128, 32, 128, 128, 0, 4.0, 0.43, 0.55, true, false},
                               {kWr64x128, 64, 128, 128, 32, 4.5, 0.46, 0.69, true, false},
                               {kWr96x128, 96, 128, 128, 64, 4.8, 0.51, 0.84, false, false},
                               {kWr128x256, 128, 256, 64, 0, 5.1, 0.53, 0.88, true, true},
                               {kWr192x256, 192, 256, 64, 128, 5.0, 0.72, 1.06, false, true}};
  // [tall][8-bit][bf16][zero term]
  static const double convert[2][2][2][2] = {{{{1.00, 1.08}, {1.04, 1.36}}, {{1.33, 1.33}, {1.35, 1.58}}},
                                             {{{1.00, 1.03}, {1.00, 1.21}}, {{1.10, 1.11}, {1.13, 1.33}}}};
  constexpr int kCUs = 256;
  const bool zero = has_zero_term(a);
  const double scales_us = 1.9 / 4096 * (a.symmetric ? 1 : 2) / a.group_size;  // per column and k
  const double mn = 1e-6 * (double)a.m * a.n;
  // us for the sums of one slice, in whole 32 x 32 tiles
  const double slice_us = 8e-6 / 5.2 * 1024 * ceil_div(a.m, 32) * ceil_div(a.n, 32);
  const double store_us = a.n % 8 != 0 ? 0.35 * mn : 0.0;
  for (const Tile& t : tiles) {
    if (a.m <= t.above || (!t.any_bits && a.bits != 4)) continue;
    const int blocks = ceil_div(a.m, t.bm) * ceil_div(a.n, t.bn);
    const int steps = ceil_div(a.k, t.step_k);
    const double c = convert[t.tall][a.bits == 8][a.t_dtype == OFQ_BF16][zero] * (a.k % t.step_k != 0 ? 1.4 : 1.0);
    const double full = t.full * (a.bits == 8 && !t.tall && a.m <= t.bm ? 1.1 : 1.0);
    auto consider = [&](int s) {
      const int per = ceil_div(steps, s);
      s = ceil_div(steps, per);  // no empty last slice
      const double us = t.start + 0.5 * mn + per * c * rounds_us(blocks * s, kCUs, t.alone, full)
                        + ceil_div(blocks * s, kCUs) * (per * t.step_k * t.bn * scales_us)
                        + (s > 1 ? 1.9 + s * slice_us : store_us);
      if (us < best) {
        best = us;
        plan->tile = t.tile;
        plan->splits = s;
      }
    };
    consider(1);
    if (!have_workspace) continue;
    // steps / s falls, the sums grow with s: least where the two are equal, or where the chip is full
    int most = kCUs / blocks < steps / 2 ? kCUs / blocks : steps / 2;
    most = most < 16 ? most : 16;
    if (most < 2) continue;
    const int s = (int)std::sqrt((steps * full * c + a.k * t.bn * scales_us) / slice_us);
    consider(s < 2 ? 2 : (s > most ? most : s));
    if (s < most) {
      consider(s < 2 ? 3 : s + 1);
      consider(most);
    }
  }
  return best;
}

// The same for gemm_core2 on the tiles and slices that launch_wq_variant takes above 64 rows.  It
// expands a code once per block where gemm_wr does once per wave: what is expanded hardly matters, and
// with 8-bit codes or a zero point and several tiles of rows it is the faster one (fp16 8-bit 700 x
// 13824 x 5120: 130 us, 177 there).
double wq_us(const LinearArgs& a, int splits) {
  const double c = (has_zero_term(a) ? 1.06 : 0.97) * (a.k % 64 != 0 ? 1.18 : 1.0);
  const int n128 = ceil_div(a.n, 128);
  double round;
  if (a.m > 128) {
    const bool wide = splits == 1 && pick_tile_width(a.m, a.n) == 192;
    const int blocks = ceil_div(a.m, 256) * (wide ? ceil_div(a.n, 192) : n128) * splits;
    round = rounds_us(blocks, 256, wide ? 1.40 : 1.02, wide ? 1.73 : 1.24);
  } else if (splits > 1) {
    round = rounds_us(n128 * splits, 256, 0.53, 0.93);
  } else if (n128 < 192) {
    round = rounds_us(ceil_div(a.n, 32), 768, 0.43, 0.90);
  } else {
    round = rounds_us(n128, 512, 0.95, 1.30);
  }
  const double mn = 1e-6 * (double)a.m * a.n;
  return 3.2 + 0.5 * mn + ceil_div(ceil_div(a.k, 64), splits) * c * round
         + (splits > 1 ? 4.1 + splits * mn * 8 / 6.5 : (a.n % 8 != 0 ? 0.2 * mn : 0.0));
}

size_t wq_partial_bytes(const LinearArgs& a) {
  const int splits = wq_splits(a);
  return splits > 1 ? (size_t)splits * (size_t)a.m * (size_t)a.n * 4 : 0;
}

// what launch_gemm_wq uses for a problem that is not gemm_wr's: the converted weight, or fp32 sums
size_t wq_bytes(const LinearArgs& a) {
  return a.m >= 1024 ? (size_t)a.n * (size_t)a.k * 2 : wq_partial_bytes(a);
}

// fp32 sums of the slices in whole 32 x 32 tiles, rounded up to whole [m, n] matrices: the unit in which
// the query has always counted slices.  Above 64 rows never less than gemm_core2's slices take, the size
// that callers know for these problems.
size_t wr_partial_bytes(const LinearArgs& a, const WrPlan& plan) {
  if (plan.splits == 1) return 0;
  const size_t mn = (size_t)a.m * (size_t)a.n * 4;
  const size_t tiles = (size_t)plan.splits * ceil_div(a.m, 32) * ceil_div(a.n, 32) * 4096;
  const size_t need = (tiles + mn - 1) / mn * mn;
  const size_t known = a.m > 64 ? wq_partial_bytes(a) : 0;
  return need > known ? need : known;
}

// Two passes for m >= 1024: the weight converted once at the rate of a large copy, and the copy-fed GEMM on it
// (within 10 % for 90 of 100 of 384 problems with m to 4096).
double two_pass_us(const LinearArgs& a) {
  const double nk = (double)a.n * a.k;
  double us;
  pick_copy_tile(a.m, a.n, a.k * 2, &us);
  return us + 2.2 + nk * (2 + a.bits / 8.0 + (a.symmetric ? 2.0 : 4.0) / a.group_size) / 5.9e6;
}

}  // namespace

// From 1024 rows on against the converted weight, with 1.1 of gemm_wr's expected time (it is 5 % short there in the
// mean): few columns or little K for the rows leave gemm_wr ahead, whose slices fill the chip and which does not write the
// weight out (1105 x 863 x 7296 fp16 8-bit 121 -> 32 us, 1024 x 4096 x 11008 4-bit 140 -> 107).  Without a
// workspace the weights of so many rows stay with gemm_core2's in-tile path.
bool gemm_wr_plan(const LinearArgs& a, bool have_workspace, WrPlan* plan) {
  if (a.m >= 1024 && !have_workspace) return false;
  const double us = wr_plan_us(a, have_workspace, plan);
  if (us >= 1e30) return false;
  if (a.m >= 1024) return us * 1.1 < two_pass_us(a);
  return a.m <= 64 || us <= wq_us(a, have_workspace ? wq_splits(a) : 1);
}

// Two passes pay once m is large: the in-tile path converts every weight tile once per 256 rows
// of x (8 times at m = 2048) and that conversion, not the MFMAs, bounds it; converting the weight
// once into the workspace and running the copy-fed GEMM on it is what the reference functor does
// for m > 8 (oneflow/core/functional/impl/quantization.cpp:341-350).  From 1024 rows on never less than the
// converted weight, the size that callers know for these problems.
size_t gemm_wq_workspace_bytes(const LinearArgs& a) {
  if (!gemm_wq_supported(a)) return 0;
  WrPlan plan;
  if (!gemm_wr_plan(a, true, &plan)) return wq_bytes(a);
  const size_t need = wr_partial_bytes(a, plan);
  return a.m >= 1024 && need < wq_bytes(a) ? wq_bytes(a) : need;
}

// The streaming kernel's rival for 16 < m <= 64: what gemm_wr is expected to take, `two_launches` us more
// if it slices K.
double gemm_wr_us(const LinearArgs& a, bool have_workspace, double two_launches) {
  WrPlan plan{kWr32x128, 1};
  const double us = wr_plan_us(a, have_workspace, &plan);
  return plan.splits > 1 ? us + two_launches : us;
}

int launch_gemm_wq(hipStream_t st, const LinearArgs& a, void* workspace, size_t workspace_bytes) {
  WrPlan plan;
  bool wr = gemm_wr_plan(a, true, &plan);
  const size_t need = wr ? wr_partial_bytes(a, plan) : wq_bytes(a);
  auto fits = [&](size_t bytes) {
    return bytes != 0 && workspace != nullptr && workspace_bytes >= bytes && ofq_aligned16(workspace);
  };
  bool have_ws = fits(need);
  if (need != 0 && !have_ws) {
    wr = gemm_wr_plan(a, false, &plan);
    have_ws = a.m >= 1024 && fits(wq_bytes(a));  // too little for the slices, enough for the converted weight
  }
  if (wr) {
    float* partials = static_cast<float*>(workspace);
    return a.t_dtype == OFQ_F16 ? launch_gemm_wr_f16(st, a, plan, partials)
                                : launch_gemm_wr_bf16(st, a, plan, partials);
  }
  if (have_ws && a.m < 1024) {
    float* partials = static_cast<float*>(workspace);
    const int splits = wq_splits(a);
    if (a.t_dtype == OFQ_F16) return launch_wq_t<f16, MfmaF16>(st, a, partials, splits);
    return launch_wq_t<bf16, MfmaBF16>(st, a, partials, splits);
  }
  if (have_ws) {
    const int rc = ofq_groupwise_dequantize(st, a.w, a.scale, a.zero, workspace,
                                            a.w_signed ? OFQ_I8 : OFQ_U8, a.t_dtype, a.bits,
                                            a.symmetric ? 1 : 0, a.n * (a.k / a.group_size),
                                            a.group_size, 1);
    if (rc != OFQ_OK) return rc;
    if (a.k % 64 != 0) {
      return a.t_dtype == OFQ_F16 ? launch_plain<true, f16, MfmaF16>(st, a, workspace)
                                  : launch_plain<true, bf16, MfmaBF16>(st, a, workspace);
    }
    if (a.t_dtype == OFQ_F16) return launch_plain<false, f16, MfmaF16>(st, a, workspace);
    return launch_plain<false, bf16, MfmaBF16>(st, a, workspace);
  }
  if (a.t_dtype == OFQ_F16) return launch_wq_t<f16, MfmaF16>(st, a, nullptr, 1);
  return launch_wq_t<bf16, MfmaBF16>(st, a, nullptr, 1);
}

// Groups along N: nothing to gain from converting inside the GEMM (a k-tile of a weight row would
// need 64 scales); above the streaming kernel's range the weight is dequantised once into the
// workspace -- the reference functor's own decomposition for m > 8,
// oneflow/core/functional/impl/quantization.cpp:341-350 -- and the copy-fed GEMM runs on it.
namespace {

// K slices of the copy-fed GEMM when its 256 x 128 tiles alone would leave most CUs without a
// block (m = 256 at n = 4096: 32 tiles): as many as fit one resident round, each >= 4 k-tiles
int gn_splits(const LinearArgs& a) {
  const int64_t blocks = ((a.m + 255) / 256) * ((a.n + 127) / 128);
  int64_t s = 256 / blocks;
  const int64_t kt = (a.k + 63) / 64;
  if (s > 8) s = 8;
  if (s > kt / 4) s = kt / 4;
  if (s < 1) s = 1;
  while (s > 1 && ((kt + s - 1) / s) * (s - 1) >= kt) --s;  // no empty last slice
  return (int)s;
}

template<typename T, class MF>
int launch_plain_split(hipStream_t st, const LinearArgs& a, const void* wt, float* partials,
                       int splits) {
  constexpr bool RG = false;  // whole k-tiles (gemm_gn_workspace_bytes)
  typedef typename TT<T>::storage S;
  BCopyParams bp;
  bp.b = static_cast<const uint8_t*>(wt);
  bp.ldb = a.k * 2;
  bp.N = (int)a.n;
  EpPartial::Params pp;
  pp.out = partials;
  const int rc = launch_core2<MF, B2Copy<RG, 128, 512>, EpPartial, 256, 128, 4, 2>(
      st, a.x, a.k * 2, bp, pp, a.m, a.n, (a.k + 63) / 64, splits);
  if (rc != OFQ_OK) return rc;
  const int64_t mn = a.m * a.n;
  const S* bias = static_cast<const S*>(a.bias);
  S* out = static_cast<S*>(a.out);
  splitk_finalize<T><<<(unsigned)((mn + 1023) / 1024), 256, 0, st>>>(partials, bias, out, (uint32_t)mn,
                                                                     (uint32_t)a.n, splits);
  return ofq_check_launch();
}

inline size_t round_up_256(size_t v) { return (v + 255) & ~(size_t)255; }

}  // namespace

// [dequantised weight n*k*sizeof(T), padded to 256 B][fp32 partial sums of the K slices, if any]
size_t gemm_gn_workspace_bytes(const LinearArgs& a) {
  if (a.group_dim != 0 || (a.t_dtype != OFQ_F16 && a.t_dtype != OFQ_BF16)) return 0;
  if (a.m <= 64 || a.k % 64 != 0 || a.n % a.group_size != 0) return 0;
  const int splits = gn_splits(a);
  return round_up_256((size_t)a.n * (size_t)a.k * 2)
         + (splits > 1 ? (size_t)splits * (size_t)a.m * (size_t)a.n * 4 : 0);
}

int launch_gemm_gn(hipStream_t st, const LinearArgs& a, void* workspace) {
  const int rc = ofq_groupwise_dequantize(st, a.w, a.scale, a.zero, workspace,
                                          a.w_signed ? OFQ_I8 : OFQ_U8, a.t_dtype, a.bits,
                                          a.symmetric ? 1 : 0, a.n / a.group_size, a.group_size,
                                          a.k);
  if (rc != OFQ_OK) return rc;
  const int splits = gn_splits(a);
  if (splits > 1) {
    float* partials = reinterpret_cast<float*>(static_cast<char*>(workspace)
                                               + round_up_256((size_t)a.n * (size_t)a.k * 2));
    if (a.t_dtype == OFQ_F16) {
      return launch_plain_split<f16, MfmaF16>(st, a, workspace, partials, splits);
    }
    return launch_plain_split<bf16, MfmaBF16>(st, a, workspace, partials, splits);
  }
  if (a.t_dtype == OFQ_F16) return launch_plain<false, f16, MfmaF16>(st, a, workspace);
  return launch_plain<false, bf16, MfmaBF16>(st, a, workspace);
}

}  // namespace ofq

using namespace ofq;

// rows of a up to which matmul_quant streams the weights whatever the shape
static constexpr int64_t kMatmulQuantRowsMaxM = 64;

namespace ofq {
namespace {

// K slices for which the workspace query makes room, the size that callers know: where the 128-wide tiles of the int8
// GEMM alone would leave most CUs without a block, as many as fit one resident round (256x128 tiles: one
// block per CU; 128x128: two), each at least 4 k-tiles of 128.
int mq_room(int64_t m, int64_t n, int64_t k) {
  const int64_t t64 = ((m + 63) / 64) * ((n + 63) / 64);
  const int64_t b256 = ((m + 255) / 256) * ((n + 127) / 128);
  const int64_t b128 = ((m + 127) / 128) * ((n + 127) / 128);
  if (m > kMatmulQuantRowsMaxM && k <= 6144) {
    if (m <= 768 && t64 >= 128 && t64 <= 768) return 1;
    if (b256 < 192 && b128 >= 192 && b128 <= 512) return 1;
  }
  // (33 to 64 rows of k >= 8192 ran as slices once: the query still makes room, the streaming kernel takes them in
  // 0.55 to 1.0 of the time, 4096 x 11008 at m = 64 26.5 -> 18.6 us)
  if (m <= (k >= 8192 ? kMatmulQuantRowsMaxM / 2 : kMatmulQuantRowsMaxM)) return 1;
  int64_t blocks = m > 128 ? b256 : b128;
  int64_t slots = m > 128 ? 256 : 512;
  // up to 512 rows on a weight with few column tiles: 128-row tiles and fewer, longer slices
  if (m <= 512 && b128 <= 128) {
    blocks = b128;
    slots = m <= 128 ? 128 : 256;
  }
  int64_t s = slots / blocks;
  const int64_t kt = (k + 127) / 128;
  if (s > 8) s = 8;
  if (s > kt / 4) s = kt / 4;
  if (s < 1) s = 1;
  while (s > 1 && ((kt + s - 1) / s) * (s - 1) >= kt) --s;  // no empty last slice
  return (int)s;
}

// Streaming kernel, tile and slices by the least expected time (kCopyCostI8), with at most `most` slices (what the
// workspace that callers know has room for): one slice on any tile, or several of 128 x 128 or 256 x 128
// tiles in one resident round, whose int32 sums and second launch cost 2 us and 1.8 to 2.3 us per 10^6 sums.
struct MqPlan {
  bool stream;
  MqTile tile;
  int splits;
};
MqPlan mq_plan(int64_t m, int64_t n, int64_t k, int most) {
  static const TileCost kSliced[2][2] = {{{128, 128, 6.47, 0.0, 0.0, 0.111, 0.430, 0.0, 0.0},
                                          {256, 128, 8.03, 0.0, 0.619, 0.185, 0.0, 0.0, 0.0}},
                                         {{128, 128, 6.29, 0.0, 0.0, 0.029, 0.614, 0.0, 0.0},
                                          {256, 128, 7.82, 0.0, 0.0, 0.065, 0.872, 0.0, 0.0}}};
  static const double kSums[2][2] = {{2.26, 1.78}, {2.22, 1.85}};  // us per 10^6 of a slice
  MqPlan plan{false, kMq64, 1};
  double best;
  const int ragged = k % 128 != 0;
  plan.tile = (MqTile)pick_tile(kCopyCostI8[ragged], kMqTiles, m, n, k, &best);
  const int64_t kt = (k + 127) / 128;
  for (int s = 2; s <= most; ++s) {
    const int64_t per = (kt + s - 1) / s;
    if (per < 2 || per * (s - 1) >= kt) continue;
    for (int i = 0; i < 2; ++i) {
      const TileCost& c = kSliced[ragged][i];
      if ((int64_t)ceil_div(m, c.bm) * ceil_div(n, c.bn) * s > 256) continue;
      const double us = tile_us(c, m, n, per, s) + kSums[ragged][i] * s * 1e-6 * (double)m * n;
      if (us < best) {
        best = us;
        plan = MqPlan{false, i == 0 ? kMq128 : kMq256x128, s};
      }
    }
  }
  if (matmul_quant_rows_supported(m, n, k)) plan.stream = matmul_quant_rows_us(m, n, k) < best;
  return plan;
}

// adds the int32 slices (integer addition: any order gives the same sum) and applies the
// epilogue of EpScale
template<typename T>
__global__ void __launch_bounds__(256)
splitk_finalize_i32(const int* __restrict__ part, const float* __restrict__ a_scale,
                    const float* __restrict__ b_scale,
                    const typename TT<T>::storage* __restrict__ bias,
                    typename TT<T>::storage* __restrict__ out, uint32_t MN, uint32_t N, int splits) {
  uint32_t i = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= MN) return;
  i = i < MN - 4 ? i : MN - 4;
  const i32x4 acc = sum_slices4<i32x4>(part + i, MN, splits);
  const float sa = a_scale[0];
  store_folded4<T>(out + i, (int)(i % N), (int)N, [&](int e, int n) {
    const float r = (float)acc[e] * (sa * b_scale[n]);
    return bias != nullptr ? r + TT<T>::load(bias + n) : r;
  });
}

template<bool RG, typename T>
int launch_mq_split(hipStream_t st, const void* a, const BCopyParams& bp, const float* a_scale,
                    const float* b_scale, const void* bias, void* out, int64_t m, int64_t n,
                    int64_t k, float* partials, const MqPlan& plan) {
  typedef typename TT<T>::storage S;
  const int splits = plan.splits;
  EpPartialI32::Params pp;
  pp.out = partials;
  int rc;
  if (plan.tile == kMq256x128) {
    rc = launch_deep<MfmaI8, RG, EpPartialI32, 256, 128, 4, 2, 3>(st, a, k, bp, pp, m, n, (k + 127) / 128, splits);
  } else {
    rc = launch_deep<MfmaI8, RG, EpPartialI32, 128, 128, 4, 2, 5>(st, a, k, bp, pp, m, n, (k + 127) / 128, splits);
  }
  if (rc != OFQ_OK) return rc;
  const int64_t mn = m * n;
  const int* pi = reinterpret_cast<const int*>(partials);
  splitk_finalize_i32<T><<<(unsigned)((mn + 1023) / 1024), 256, 0, st>>>(
      pi, a_scale, b_scale, static_cast<const S*>(bias), static_cast<S*>(out), (uint32_t)mn, (uint32_t)n,
      splits);
  return ofq_check_launch();
}

// one launch, no K slices
template<bool RG, typename T>
int launch_mq(hipStream_t st, const void* a, const BCopyParams& bp, const float* a_scale,
              const float* b_scale, const void* bias, void* out, int64_t m, int64_t n, int64_t k,
              MqTile tile) {
  typedef EpScale<T> EP;
  typename EP::Params ep;
  ep.a_scale = a_scale;
  ep.b_scale = b_scale;
  ep.bias = static_cast<const typename TT<T>::storage*>(bias);
  ep.out = static_cast<typename TT<T>::storage*>(out);
  const int64_t kt = (k + 127) / 128;
  switch (tile) {
    case kMq64: return launch_deep<MfmaI8, RG, EP, 64, 64, 2, 2, 5>(st, a, k, bp, ep, m, n, kt);
    case kMq64Short: return launch_deep<MfmaI8, RG, EP, 64, 64, 2, 2, 3>(st, a, k, bp, ep, m, n, kt);
    case kMq128x64: return launch_deep<MfmaI8, RG, EP, 128, 64, 4, 2, 6>(st, a, k, bp, ep, m, n, kt);
    case kMq128x64Short: return launch_deep<MfmaI8, RG, EP, 128, 64, 4, 2, 3>(st, a, k, bp, ep, m, n, kt);
    case kMq128: return launch_deep<MfmaI8, RG, EP, 128, 128, 4, 2, 5>(st, a, k, bp, ep, m, n, kt);
    case kMq128Short: return launch_core2<MfmaI8, B2Copy<RG, 128, 512>, EP, 128, 128, 4, 2>(st, a, k, bp, ep, m, n, kt);
    case kMq256x128: return launch_deep<MfmaI8, RG, EP, 256, 128, 4, 2, 3>(st, a, k, bp, ep, m, n, kt);
    default: break;
  }
  if constexpr (RG) {  // (why: launch_pp)
    if (tile == kMq256x192) {
      return launch_core2<MfmaI8, B2Copy<RG, 192, 512>, EP, 256, 192, 4, 2>(st, a, k, bp, ep, m, n, kt);
    }
  }
  const int width = kCopyCostI8[RG][tile].bn;
  return launch_gemm_pp_i8(st, a, bp.b, a_scale, b_scale, bias, out, TT<T>::dtype, m, n, k, width);
}

}  // namespace
}  // namespace ofq

extern "C" size_t ofq_matmul_quant_workspace_bytes(int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  const int splits = ofq::mq_room(m, n, k);
  return splits > 1 ? (size_t)splits * (size_t)m * (size_t)n * 4 : 0;
}

extern "C" int ofq_matmul_quant_ws(void* stream, const void* a, const void* b, const float* a_scale,
                                   const float* b_scale, const void* bias, void* out, int out_dtype,
                                   int64_t m, int64_t n, int64_t k, void* workspace,
                                   size_t workspace_bytes);

extern "C" int ofq_matmul_quant(void* stream, const void* a, const void* b, const float* a_scale,
                                const float* b_scale, const void* bias, void* out, int out_dtype,
                                int64_t m, int64_t n, int64_t k) {
  return ofq_matmul_quant_ws(stream, a, b, a_scale, b_scale, bias, out, out_dtype, m, n, k, nullptr,
                             0);
}

extern "C" int ofq_matmul_quant_ws(void* stream, const void* a, const void* b, const float* a_scale,
                                   const float* b_scale, const void* bias, void* out, int out_dtype,
                                   int64_t m, int64_t n, int64_t k, void* workspace,
                                   size_t workspace_bytes) {
  OFQ_RETURN_IF(out_dtype != OFQ_F16 && out_dtype != OFQ_BF16 && out_dtype != OFQ_F32,
                OFQ_ERR_BAD_DTYPE);
  OFQ_RETURN_IF(m < 0 || n < 0 || k <= 0, OFQ_ERR_BAD_SHAPE);
  if (m == 0 || n == 0) return OFQ_OK;
  const int64_t i32max = 0x7FFFFFFF;
  OFQ_RETURN_IF(m * k > i32max || n * k > i32max || m * n > i32max, OFQ_ERR_UNSUPPORTED);
  // rows are consumed in 64-byte chunks of K (streaming kernel) or 128-byte tiles (GEMM, the last
  // one padded with zeros)
  OFQ_RETURN_IF(k % 64 != 0, OFQ_ERR_UNSUPPORTED);
  OFQ_RETURN_IF(a == nullptr || b == nullptr || a_scale == nullptr || b_scale == nullptr
                    || out == nullptr,
                OFQ_ERR_NULL_POINTER);
  OFQ_RETURN_IF(!ofq_aligned16(a) || !ofq_aligned16(b) || !ofq_aligned16(out), OFQ_ERR_MISALIGNED);
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto stream_weights = [&] {
    return launch_matmul_quant_rows(st, a, b, a_scale, b_scale, bias, out, out_dtype, m, n, k);
  };
  // few rows of a: the weights stream once (above 64 rows where that is expected to be faster)
  if (m <= kMatmulQuantRowsMaxM && matmul_quant_rows_supported(m, n, k)) return stream_weights();
  BCopyParams bp;
  bp.b = static_cast<const uint8_t*>(b);
  bp.ldb = k;
  bp.N = (int)n;
  const int room = mq_room(m, n, k);
  const size_t need = (size_t)room * (size_t)m * (size_t)n * 4;
  const bool slices = room > 1 && workspace != nullptr && workspace_bytes >= need && ofq_aligned16(workspace);
  const MqPlan plan = mq_plan(m, n, k, slices ? room : 1);
  if (plan.stream) return stream_weights();
  if (plan.splits > 1) {
    float* part = static_cast<float*>(workspace);
#define OFQ_MQS(RG, T)                                                                           \
  return launch_mq_split<RG, T>(st, a, bp, a_scale, b_scale, bias, out, m, n, k, part, plan)
    if (k % 128 != 0) {
      switch (out_dtype) {
        case OFQ_F16: OFQ_MQS(true, f16);
        case OFQ_BF16: OFQ_MQS(true, bf16);
        default: OFQ_MQS(true, float);
      }
    }
    switch (out_dtype) {
      case OFQ_F16: OFQ_MQS(false, f16);
      case OFQ_BF16: OFQ_MQS(false, bf16);
      default: OFQ_MQS(false, float);
    }
#undef OFQ_MQS
  }
  if (k % 128 != 0) {
    switch (out_dtype) {
      case OFQ_F16: return launch_mq<true, f16>(st, a, bp, a_scale, b_scale, bias, out, m, n, k, plan.tile);
      case OFQ_BF16: return launch_mq<true, bf16>(st, a, bp, a_scale, b_scale, bias, out, m, n, k, plan.tile);
      default: return launch_mq<true, float>(st, a, bp, a_scale, b_scale, bias, out, m, n, k, plan.tile);
    }
  }
  switch (out_dtype) {
    case OFQ_F16: return launch_mq<false, f16>(st, a, bp, a_scale, b_scale, bias, out, m, n, k, plan.tile);
    case OFQ_BF16: return launch_mq<false, bf16>(st, a, bp, a_scale, b_scale, bias, out, m, n, k, plan.tile);
    default: return launch_mq<false, float>(st, a, bp, a_scale, b_scale, bias, out, m, n, k, plan.tile);
  }
}
