// Decode kernel of fused_linear_with_groupwise_quantized_weight for every 16-bit element type
// and both code widths, with x kept in its natural order.
//
// Same row split as gemv_w4p_f16 (a whole number of blocks per CU, each owning consecutive
// weight rows that it walks as 16-row tiles; the m <= 16 rows of x ride as the first operand of
// a 16x16x32 MFMA, so the weights stream from HBM once whatever m is), but the codes are
// expanded to T in natural element order by dequant8_b4 / dequant16_b8:
//   w~ = T(T(q) * s) + z  with the reference's roundings
//   (oneflow/user/kernels/groupwise_quantization_kernels.cu:73-117, :582-642),
// so bf16 (whose products have to be rounded in fp32 arithmetic: there is no packed bf16 math)
// and 8-bit codes get the same treatment as the fp16 4-bit case.  Groups may be as short as one
// lane's 16 bytes of codes (32 4-bit or 16 8-bit elements).
//
// K is any multiple of a lane's share of a chunk (LK = 32 4-bit or 16 8-bit elements), so a lane's
// share lies inside or outside the row as a whole.  In the last chunk of a ragged row (a K shard
// of 43 groups of 64, say) the lanes beyond K re-read the row's first bytes, expand them with a scale
// and a zero point of 0 (a w~ that overflows T would turn the zero of x it meets into NaN) and meet
// zeros of x: nothing out of bounds is read and their products add 0.  Before, such rows went to the
// one-wave-per-row fallback (2 layers of 4352 / 14624 columns, groups of 32, 3 rows of x: 836 us).
#pragma once

#include "dequant_regs.h"
#include "gemv_kernels.h"
#include "ofq_device.h"
#include "ofq_internal.h"
#include "scale_panel.h"

namespace ofq {
namespace {

constexpr int kRowsMaxTiles = 4;   // 16-row tiles per block
constexpr int kRowsMaxUnits = 8;   // 16-byte pieces of x a thread may stage

template<typename T>
struct MfmaK32;
template<>
struct MfmaK32<f16> {
  static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template<>
struct MfmaK32<bf16> {
  static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};

// raw bits of a T -> float at the point of use (keeps the load's wait where the value is needed)
template<typename T>
__device__ __forceinline__ float raw16_at_end(uint16_t raw) {
  uint32_t v = raw;
  asm volatile("" : "+v"(v));
  if constexpr (TT<T>::dtype == OFQ_BF16) {
    return __builtin_bit_cast(float, v << 16);
  } else {
    return (float)__builtin_bit_cast(f16, (uint16_t)v);
  }
}

// STAGED: x is copied to LDS once per block (m * k small enough); otherwise every wave reads the
// x of its chunk pairs straight from global memory (x stays in L2: it is re-read by every block).
// Either way a wave takes chunk pairs p = wave, wave + NWAVES, ... and walks all tiles of the
// block for each, so x is fetched once per pair and the per-tile sums stay in registers.
template<typename T, int BITS, bool SIGNED, int ZMODE, int NWAVES, bool STAGED>
__device__ __forceinline__ void
gemv_rows_body(int block, const uint16_t* __restrict__ x, const uint8_t* __restrict__ w,
               const uint16_t* __restrict__ scale, const uint16_t* __restrict__ zero,
               const uint16_t* __restrict__ bias, uint16_t* __restrict__ out, int M, int N, int K,
               int group_size, int gs_shift, int rows_per_block) {
  typedef typename TT<T>::storage S;
  static_assert(sizeof(S) == 2, "16-bit element types");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int NT = NWAVES * 64;
  constexpr int CK = BITS == 4 ? 128 : 64;  // elements per chunk: 64 bytes of codes per row
  constexpr int LK = CK / 4;                // elements per lane and chunk
  constexpr int XV = LK / 8;                // 16-byte pieces of x per lane and chunk
  const int nchunks = (K + CK - 1) / CK;
  const int npairs = (nchunks + 1) >> 1;
  const int row_bytes = K / LK * 16;
  const int G = K / group_size;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15;
  const int kb = lane >> 4;
  const int row0 = block * rows_per_block;
  int rows_blk = N - row0;
  if (rows_blk > rows_per_block) rows_blk = rows_per_block;
  if (rows_blk <= 0) return;
  const int ntiles = (rows_blk + 15) >> 4;
  const bool has_x = r < M;

  // LDS: [scales rows_per_block*G, padded to 16 B][zeros, same size (asymmetric only)]
  //      [64 zero bytes][x: M rows of K*2+16 bytes (STAGED)]; the sums of the waves
  //      (tiles*NWAVES*M*16 f32) take the place of x once every wave has walked its pairs
  const int tile_bytes = (rows_per_block * G * 2 + 15) & ~15;
  uint16_t* sl = reinterpret_cast<uint16_t*>(smem);
  uint16_t* zl = reinterpret_cast<uint16_t*>(reinterpret_cast<uint8_t*>(sl) + tile_bytes);
  uint8_t* zrec = reinterpret_cast<uint8_t*>(sl) + (ZMODE == kZeroAsym ? 2 : 1) * tile_bytes;
  uint8_t* xs = zrec + 64;
  float* red = reinterpret_cast<float*>(xs);
  const int x_pitch = K * 2 + 16;  // rows skewed by 16 bytes: lanes of different m reading the
                                   // same k hit different LDS bank groups

  // ---- requests that feed LDS go out first ----------------------------------------------------
  const int upr = K >> 3;  // 16-byte pieces per row of x
  const int nunits = M * upr;
  u32x4 xu[kRowsMaxUnits];
  if (STAGED) {
#pragma unroll
    for (int i = 0; i < kRowsMaxUnits; ++i) {
      if (wave * 64 + i * NT >= nunits) break;
      const int u = tid + i * NT;
      if (u < nunits) xu[i] = *reinterpret_cast<const u32x4*>(x + (int64_t)u * 8);
    }
  }
  const int tile_halves = rows_blk * G;
  const uint16_t* stile = scale + (int64_t)row0 * G;
  const bool s_aligned = ((reinterpret_cast<uintptr_t>(stile)) & 15u) == 0;
  const uint16_t* ztile = ZMODE == kZeroAsym ? zero + (int64_t)row0 * G : stile;
  u32x4 sreg, zreg;
  const int se = tid * 8;
  const bool s_vec = s_aligned && se + 8 <= tile_halves;
  if (s_vec) {
    sreg = *reinterpret_cast<const u32x4*>(stile + se);
    if (ZMODE == kZeroAsym) zreg = *reinterpret_cast<const u32x4*>(ztile + se);
  }
  // bias of the first output this thread folds at the end: tid = (tile * M + m) * 16 + n
  uint16_t bias_raw = 0;
  {
    const int t = tid / (M * 16);
    const int row_l = t * 16 + (tid & 15);
    if (bias != nullptr && t < ntiles && row_l < rows_blk) bias_raw = bias[row0 + row_l];
  }

  // ---- codes of (tile, pair): one 16-byte load per lane and chunk ------------------------------
  const uint8_t* wbase = w + (int64_t)row0 * row_bytes;
  // Straight-line on purpose: a load under a branch makes the compiler wait for everything in
  // flight at the first LDS fill.  A slot without an item reads one and the same 16 bytes in
  // every lane; lanes past the block's rows re-read its first row (never stored).
  auto issue = [&](int tile, int pair, u32x4 (&dst)[2], bool live) {
    const int row_l = tile * 16 + r;
    const bool ok = row_l < rows_blk;
    const uint8_t* p = wbase + (int64_t)(ok ? row_l : 0) * row_bytes;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int off = (2 * pair + u) * 64 + kb * 16;
      const uint8_t* q = p + (off < row_bytes ? off : 0);
      dst[u] = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4*>(live ? q : w + (int64_t)row0 * row_bytes));
    }
  };
  int pair = wave;
  u32x4 wq[2];
  {
    const bool live = pair < npairs;
    issue(0, live ? pair : 0, wq, live);
  }

  // ---- fill LDS -------------------------------------------------------------------------------
  if (s_vec) {
    *reinterpret_cast<u32x4*>(sl + se) = sreg;
    if (ZMODE == kZeroAsym) *reinterpret_cast<u32x4*>(zl + se) = zreg;
  } else if (se < tile_halves && s_aligned) {
    for (int j = se; j < tile_halves && j < se + 8; ++j) {
      sl[j] = stile[j];
      if (ZMODE == kZeroAsym) zl[j] = ztile[j];
    }
  }
  for (int e = (s_aligned ? NT * 8 : 0) + tid; e < tile_halves; e += NT) {
    sl[e] = stile[e];
    if (ZMODE == kZeroAsym) zl[e] = ztile[e];
  }
  if (STAGED) {
    if (tid < 16) reinterpret_cast<uint32_t*>(zrec)[tid] = 0u;
    // piece u of x lies in row u / upr; rows advance by (NT / upr, NT % upr) per step
    const int qstep = NT / upr, rstep = NT - qstep * upr;
    int xrow = tid / upr, xrem = tid - xrow * upr;
#pragma unroll
    for (int i = 0; i < kRowsMaxUnits; ++i) {
      if (wave * 64 + i * NT >= nunits) break;
      if (tid + i * NT < nunits) {
        *reinterpret_cast<u32x4*>(xs + (size_t)xrow * x_pitch + xrem * 16) = xu[i];
      }
      xrow += qstep;
      xrem += rstep;
      if (xrem >= upr) {
        xrem -= upr;
        ++xrow;
      }
    }
  }
  __syncthreads();

  // this lane's 2 * LK bytes of x per chunk: row r, k-slot kb.  Lanes r >= M feed rows of the
  // product that are never stored: a zero record (STAGED) or row 0 again (same addresses as the
  // lanes of r = 0, no extra traffic).
  const uint8_t* xlane;
  int xstride = CK * 2;
  if (STAGED) {
    xlane = has_x ? xs + (size_t)r * x_pitch + kb * (LK * 2) : zrec;
    if (!has_x) xstride = 0;
  } else {
    xlane = reinterpret_cast<const uint8_t*>(x) + ((size_t)(has_x ? r : 0) * K + kb * LK) * 2;
  }
  f32x4 acc[kRowsMaxTiles][2];
#pragma unroll
  for (int t = 0; t < kRowsMaxTiles; ++t) {
    acc[t][0] = f32x4{0.f, 0.f, 0.f, 0.f};
    acc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  while (pair < npairs) {
    u32x4 xa[2][XV];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = 2 * pair + u;
      const bool in_row = c * CK + kb * LK < K;
      if (STAGED) {
        const u32x4* xp = reinterpret_cast<const u32x4*>(in_row ? xlane + (size_t)c * xstride : zrec);
#pragma unroll
        for (int j = 0; j < XV; ++j) xa[u][j] = xp[j];
      } else {
        const u32x4* xp = reinterpret_cast<const u32x4*>(xlane + (size_t)(in_row ? c : 0) * xstride
                                                         - (in_row ? 0 : kb * LK * 2));
#pragma unroll
        for (int j = 0; j < XV; ++j) xa[u][j] = xp[j];
        if ((c + 1) * CK > K) {  // (the same for every lane: the last chunk of a ragged row)
#pragma unroll
          for (int j = 0; j < XV; ++j) xa[u][j] = in_row ? xa[u][j] : u32x4{0u, 0u, 0u, 0u};
        }
      }
    }
#pragma unroll
    for (int t = 0; t < kRowsMaxTiles; ++t) {
      if (t < ntiles) {
        const int srow = (t * 16 + r) * G;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int c = 2 * pair + u;
          if (c < nchunks) {
            int k0 = c * CK + kb * LK;
            const bool in_row = k0 < K;
            k0 = in_row ? k0 : 0;
            const int grp = gs_shift >= 0 ? (k0 >> gs_shift) : (k0 / group_size);
            float s = TT<T>::load(reinterpret_cast<const S*>(sl) + srow + grp);
            float z = 0.f;
            if (ZMODE == kZeroAsym) z = TT<T>::load(reinterpret_cast<const S*>(zl) + srow + grp);
            s = in_row ? s : 0.f;
            z = in_row ? z : 0.f;
            if (ZMODE == kZeroSymU) z = TT<T>::round(-(float)((1 << (BITS - 1)) - 1) * s);
            if constexpr (BITS == 4) {
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                const u32x4 b = dequant8_b4<T, SIGNED, ZMODE>(wq[u][j], s, z);
                // two accumulators: consecutive MFMAs do not wait for each other
                acc[t][j & 1] = MfmaK32<T>::mma(xa[u][j], b, acc[t][j & 1]);
              }
            } else {
              u32x4 b0, b1;
              dequant16_b8<T, SIGNED, ZMODE>(wq[u], s, z, b0, b1);
              acc[t][0] = MfmaK32<T>::mma(xa[u][0], b0, acc[t][0]);
              acc[t][1] = MfmaK32<T>::mma(xa[u][1], b1, acc[t][1]);
            }
          }
        }
        // codes of the next item: the next tile of this pair, else tile 0 of the wave's next pair
        const bool last_t = t + 1 >= ntiles;
        const int np = last_t ? pair + NWAVES : pair;
        const bool live = np < npairs;
        issue(last_t ? 0 : t + 1, live ? np : 0, wq, live);
      }
    }
    pair += NWAVES;
  }
  // every wave writes its sums of every tile (zeros when it had no pair) where x was
  if (STAGED) __syncthreads();  // ... which every wave has finished reading
#pragma unroll
  for (int t = 0; t < kRowsMaxTiles; ++t) {
    if (t < ntiles) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = 4 * kb + v;
        if (m < M) red[((t * NWAVES + wave) * M + m) * 16 + r] = acc[t][0][v] + acc[t][1][v];
      }
    }
  }
  __syncthreads();
  const int nout = ntiles * M * 16;
  for (int o = tid; o < nout; o += NT) {
    const int t = o / (M * 16);
    const int rem = o - t * (M * 16);  // m * 16 + n
    float sum = 0.f;
#pragma unroll
    for (int wv = 0; wv < NWAVES; ++wv) sum += red[(t * NWAVES + wv) * M * 16 + rem];
    const int m = rem >> 4;
    const int row_l = t * 16 + (rem & 15);
    if (row_l < rows_blk) {
      float bv;
      if (o == tid) {
        bv = raw16_at_end<T>(bias_raw);
      } else {
        bv = bias != nullptr ? TT<T>::load(reinterpret_cast<const S*>(bias) + row0 + row_l) : 0.f;
      }
      TT<T>::store(reinterpret_cast<S*>(out) + (int64_t)m * N + row0 + row_l, sum + bv);
    }
  }
}

template<typename T, int BITS, bool SIGNED, int ZMODE, int NWAVES, bool STAGED>
__global__ void __launch_bounds__(NWAVES * 64)
gemv_rows(const uint16_t* __restrict__ x, const uint8_t* __restrict__ w,
          const uint16_t* __restrict__ scale, const uint16_t* __restrict__ zero,
          const uint16_t* __restrict__ bias, uint16_t* __restrict__ out, int M, int N, int K,
          int group_size, int gs_shift, int rows_per_block) {
  gemv_rows_body<T, BITS, SIGNED, ZMODE, NWAVES, STAGED>(blockIdx.x, x, w, scale, zero, bias, out,
                                                         M, N, K, group_size, gs_shift,
                                                         rows_per_block);
}

// Several linears of the same m, k and quantisation in one launch (q/k/v, gate/up ...): the grid
// is the concatenation of the problems' blocks, every problem cut into rows_per_block-row
// blocks; a block finds its problem in the table and runs the single-problem body on it.
template<typename T, int BITS, bool SIGNED, int ZMODE, int NWAVES, bool STAGED>
__global__ void __launch_bounds__(NWAVES * 64)
gemv_rows_grouped(GemvGroup g, int M, int K, int group_size, int gs_shift, int rows_per_block) {
  const GemvProblem pr = select_problem(g, (int)blockIdx.x);
  gemv_rows_body<T, BITS, SIGNED, ZMODE, NWAVES, STAGED>(
      (int)blockIdx.x - pr.first_block, static_cast<const uint16_t*>(pr.x), pr.w,
      static_cast<const uint16_t*>(pr.scale), static_cast<const uint16_t*>(pr.zero),
      static_cast<const uint16_t*>(pr.bias), static_cast<uint16_t*>(pr.out), M, pr.N, K,
      group_size, gs_shift, rows_per_block);
}

// ---------------------------------------------------------------------------------------------
// 16 < m <= 64: the same row split with MT = 2, 3 or 4 sixteen-row tiles of x per MFMA group.  A
// weight tile is expanded once per chunk and meets all MT tiles of x, which come from L2 chunk
// by chunk (x is far too large for LDS here: m * k * 2 bytes per block); a wave walks chunks
// c = wave, wave + NWAVES, ... and, per chunk, every 16-row weight tile of the block.  Sums stay in
// registers and are folded through LDS one weight tile at a time.  No barrier inside the k loop.
//
// What bounds it: no unit of the chip, but two waves a SIMD that wait.  At 48 x 11008 x 4096 (fp16, zero
// point, 17.9 us) a wave waits for memory 36 % of its life and for an issue slot 33 %; the vector units are
// busy 42 % of the time, LDS 23 %, the matrix cores 12 %, and L2 hands out about 9 TB/s (every block reads all
// of x: 100 MB).  A chunk costs a wave its turn through request, LDS, conversion and product whatever m
// is, so the time follows the chunks per wave (64 x 4096 x 11008 fp16: 27.6 us for 23 MB of weights); the
// dispatch leaves long rows of weights to gemm_wr for that.  Everything a chunk needs, its MT * 16 rows x 2 CK
// bytes of x and its NTL weight tiles, is requested while the chunk before is worked on (one weight tile
// in flight took 20.3 us at 64 x 11008 x 4096 where this takes 19.0, and 26.1 against 21.2 at 48 rows
// of 8-bit codes).  The requests are unconditional and straight line (a tile past the block's rows
// re-reads its first row in every lane: one cached line), which keeps the compiler's wait counts exact.
//
// x.  A lane's operand of x is 16 bytes out of a 64-byte run of one of 16 rows, so a wave-level
// request straight from global memory would touch 64 cache lines for 1 KB of data and the vector
// cache's tag rate would bound the kernel.  A wave requests x with neighbouring lanes on
// neighbouring bytes (8 cache lines per request), parks the chunk in a buffer of its own in LDS
// (rows padded by 16 bytes) and reads its operands from there.  The buffers share their memory with
// the reduction area, which is used only after the k loop.
//
// Scales.  The scales (and zeros) of the block's rows are copied to LDS for panel_chunks chunks at a
// time: all of K unless long rows of short groups leave no room for it.  A row of the panel ends with a
// zero, the scale of a lane past the end of K.
// ---------------------------------------------------------------------------------------------
struct RowsMat {  // a weight and what belongs to it
  const uint8_t* w;
  const uint16_t* scale;
  const uint16_t* zero;
  const uint16_t* bias;
  uint16_t* out;
};
inline RowsMat rows_mat(const LinearArgs& a) {
  return RowsMat{static_cast<const uint8_t*>(a.w), static_cast<const uint16_t*>(a.scale),
                 static_cast<const uint16_t*>(a.zero), static_cast<const uint16_t*>(a.bias),
                 static_cast<uint16_t*>(a.out)};
}
inline void fill_group(GemvGroup& g, const LinearArgs* pr, int count, int rpb) {
  g.count = count;
  int first = 0;
  for (int i = 0; i < count; ++i) {
    g.p[i].x = pr[i].x;
    g.p[i].w = static_cast<const uint8_t*>(pr[i].w);
    g.p[i].scale = pr[i].scale;
    g.p[i].zero = pr[i].zero;
    g.p[i].bias = pr[i].bias;
    g.p[i].out = pr[i].out;
    g.p[i].N = (int)pr[i].n;
    g.p[i].first_block = first;
    first += (int)((pr[i].n + rpb - 1) / rpb);
  }
}

template<int BITS, int MT>
struct RowsMtX {
  static constexpr int CK = BITS == 4 ? 128 : 64;
  static constexpr int kRowBytes = CK * 2;           // of x per row and chunk
  static constexpr int kPitch = kRowBytes + 16;      // in LDS
  static constexpr int kLanesPerRow = kRowBytes / 16;
  static constexpr int kRowsPerReq = 64 / kLanesPerRow;
  static constexpr int kReqs = MT * 16 / kRowsPerReq;
  static constexpr int kWaveBytes = MT * 16 * kPitch;
};

// NTL: weight tiles of a matrix in a block; NMAT = 2: the two weights of a gated unit, whose blocks own the same
// rows of both and form y = hidden * act(gate) from the rounded sums.  One launch for q/k/v or for a gated unit
// instead of one each and the gating's: 5840 random layers of 17 to 64 rows of x (k 1024 to 6000) take 1 / 2.35
// of the time for three linears of k, k/c, k/c rows (each alone is bound by its launch and one short turn
// of the waves), 7 300 gated units 1 / 1.28 (those of 100 MB and more the same).  Where that is expected to
// take longer than one by one (3 % of the gated units): launch_gemv_mt_several.
template<typename T, int BITS, bool SIGNED, int ZMODE, int NWAVES, int MT, int NTL, int NMAT>
__device__ __forceinline__ void
gemv_rows_mt_body(int block, const uint16_t* __restrict__ x, const RowsMat (&mats)[NMAT], int N,
                  uint16_t* __restrict__ y, int act, int M, int K, int group_size, int gs_shift,
                  int rows_per_block, int panel_chunks, int panel_groups) {
  typedef typename TT<T>::storage S;
  static_assert(sizeof(S) == 2, "16-bit element types");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int NT = NWAVES * 64;
  constexpr int CK = BITS == 4 ? 128 : 64;
  constexpr int LK = CK / 4;
  const int nchunks = (K + CK - 1) / CK;
  const int row_bytes = K / LK * 16;
  const int G = K / group_size;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15;
  const int kb = lane >> 4;
  const int row0 = block * rows_per_block;
  int rows_blk = N - row0;
  if (rows_blk > rows_per_block) rows_blk = rows_per_block;
  if (rows_blk <= 0) return;
  const int ntiles = (rows_blk + 15) >> 4;

  // LDS: [the waves' x buffers | red NWAVES*MT*256 f32][scales rows_per_block*(panel_groups + 1),
  //      padded to 16 B, of every matrix][zeros (asymmetric)]
  typedef RowsMtX<BITS, MT> XB;
  float* red = reinterpret_cast<float*>(smem);
  const int pitch = panel_groups + 1;
  const int panel_bytes = (rows_per_block * pitch * 2 + 15) & ~15;
  constexpr size_t kRedBytes = (size_t)NWAVES * MT * 256 * 4;
  constexpr size_t kFront = (size_t)NWAVES * XB::kWaveBytes > kRedBytes
                                ? (size_t)NWAVES * XB::kWaveBytes : kRedBytes;
  uint16_t* sl = reinterpret_cast<uint16_t*>(smem + kFront);
  const int panel = panel_bytes / 2;  // 16-bit values from one matrix's to the next one's
  uint16_t* zl = sl + NMAT * panel;
  uint8_t* xbuf = smem + (size_t)wave * XB::kWaveBytes;

  const uint8_t* wblk[NMAT];
#pragma unroll
  for (int mat = 0; mat < NMAT; ++mat) wblk[mat] = mats[mat].w + (int64_t)row0 * row_bytes;
  uint32_t roff[NTL];  // of this lane's row of every tile
#pragma unroll
  for (int t = 0; t < NTL; ++t) {
    const int row_l = t * 16 + r;
    roff[t] = row_l < rows_blk ? (uint32_t)row_l * (uint32_t)row_bytes : 0u;
  }
  auto request_codes = [&](int c, u32x4 (&dst)[NMAT * NTL]) {  // (a chunk past the end re-reads chunk 0)
    int off = c * 64 + kb * 16;
    off = off < row_bytes ? off : 0;
#pragma unroll
    for (int t = 0; t < NMAT * NTL; ++t) {
      dst[t] = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4*>(wblk[t / NTL] + roff[t % NTL] + (uint32_t)off));
    }
  };
  // request i of a chunk covers rows kRowsPerReq * i + lane / kLanesPerRow, 16 bytes per lane; rows
  // >= M feed outputs never stored and re-read row 0
  const int xpiece = (lane % XB::kLanesPerRow) * 16;
  uint32_t xoff[XB::kReqs];
#pragma unroll
  for (int i = 0; i < XB::kReqs; ++i) {
    const int row = i * XB::kRowsPerReq + lane / XB::kLanesPerRow;
    xoff[i] = (uint32_t)(row < M ? row : 0) * (uint32_t)(K * 2);
  }
  u32x4 xg[XB::kReqs];
  auto request_x = [&](int c) {
    int off = c * XB::kRowBytes + xpiece;
    off = off < K * 2 ? off : 0;
#pragma unroll
    for (int i = 0; i < XB::kReqs; ++i) {
      xg[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(x) + xoff[i]
                                              + (uint32_t)off);
    }
  };
  f32x4 acc[NMAT * NTL][MT];
#pragma unroll
  for (int t = 0; t < NMAT * NTL; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

  int c = wave;
  u32x4 code_a[NMAT * NTL], code_b[NMAT * NTL];
  request_x(c);
  request_codes(c, code_a);

  int g0 = 0;  // first group of the panel
  auto fill_panel = [&](int first_chunk) {
    g0 = gs_shift >= 0 ? (first_chunk * CK) >> gs_shift : (first_chunk * CK) / group_size;
    const int ng = G - g0 < panel_groups ? G - g0 : panel_groups;
#pragma unroll
    for (int mat = 0; mat < NMAT; ++mat) {
      const uint16_t* sblk = mats[mat].scale + (int64_t)row0 * G + g0;
      const uint16_t* zblk = ZMODE == kZeroAsym ? mats[mat].zero + (int64_t)row0 * G + g0 : sblk;
      copy_scale_panel<NT, ZMODE == kZeroAsym, false>(sblk, zblk, G, rows_blk, rows_blk, ng, pitch,
                                                      sl + mat * panel, zl + mat * panel, tid);
      if (tid < rows_per_block) {  // (at most 64 rows)
        sl[mat * panel + tid * pitch + panel_groups] = 0;
        if (ZMODE == kZeroAsym) zl[mat * panel + tid * pitch + panel_groups] = 0;
      }
    }
    __syncthreads();
  };

  auto work = [&](const u32x4 (&cur)[NMAT * NTL], u32x4 (&nxt)[NMAT * NTL]) {
    const int k0 = c * CK + kb * LK;
    if ((c + 1) * CK > K) {  // (the same for every lane: the last chunk of a ragged row)
#pragma unroll
      for (int i = 0; i < XB::kReqs; ++i) {
        xg[i] = c * XB::kRowBytes + xpiece < K * 2 ? xg[i] : u32x4{0u, 0u, 0u, 0u};
      }
    }
    // the wave's own buffer: its LDS operations retire in order, so these stores cannot pass the
    // operand reads of the chunk before
#pragma unroll
    for (int i = 0; i < XB::kReqs; ++i) {
      const int row = i * XB::kRowsPerReq + lane / XB::kLanesPerRow;
      *reinterpret_cast<u32x4*>(xbuf + row * XB::kPitch + xpiece) = xg[i];
    }
    request_x(c + NWAVES);
    request_codes(c + NWAVES, nxt);
    int grp = (gs_shift >= 0 ? (k0 >> gs_shift) : (k0 / group_size)) - g0;
    grp = k0 < K ? grp : panel_groups;
    float s[NMAT * NTL], z[NMAT * NTL];
#pragma unroll
    for (int t = 0; t < NMAT * NTL; ++t) {
      const int at = t / NTL * panel + (t % NTL * 16 + r) * pitch + grp;
      s[t] = TT<T>::load(reinterpret_cast<const S*>(sl) + at);
      z[t] = 0.f;
      if (ZMODE == kZeroAsym) z[t] = TT<T>::load(reinterpret_cast<const S*>(zl) + at);
      if (ZMODE == kZeroSymU) z[t] = TT<T>::round(-(float)((1 << (BITS - 1)) - 1) * s[t]);
    }
    const uint8_t* xl = xbuf + r * XB::kPitch + kb * (LK * 2);
    if constexpr (BITS == 4) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        u32x4 xa[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          xa[mt] = *reinterpret_cast<const u32x4*>(xl + mt * 16 * XB::kPitch + j * 16);
        }
#pragma unroll
        for (int t = 0; t < NMAT * NTL; ++t) {
          if (t % NTL < ntiles) {
            const u32x4 b = dequant8_b4<T, SIGNED, ZMODE>(cur[t][j], s[t], z[t]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[t][mt] = MfmaK32<T>::mma(xa[mt], b, acc[t][mt]);
          }
        }
      }
    } else {
      u32x4 xa[MT][2];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        xa[mt][0] = *reinterpret_cast<const u32x4*>(xl + mt * 16 * XB::kPitch);
        xa[mt][1] = *reinterpret_cast<const u32x4*>(xl + mt * 16 * XB::kPitch + 16);
      }
#pragma unroll
      for (int t = 0; t < NMAT * NTL; ++t) {
        if (t % NTL < ntiles) {
          u32x4 b0, b1;
          dequant16_b8<T, SIGNED, ZMODE>(cur[t], s[t], z[t], b0, b1);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[t][mt] = MfmaK32<T>::mma(xa[mt][0], b0, acc[t][mt]);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[t][mt] = MfmaK32<T>::mma(xa[mt][1], b1, acc[t][mt]);
        }
      }
    }
    c += NWAVES;
  };
  for (int first = 0; first < nchunks; first += panel_chunks) {
    if (first > 0) __syncthreads();  // every wave is done with the panel before
    fill_panel(first);
    const int last = nchunks - first < panel_chunks ? nchunks : first + panel_chunks;
    // (panel_chunks is a multiple of 2 * NWAVES: every wave enters a panel with its codes in code_a)
    while (c < last) {
      work(code_a, code_b);
      if (c >= last) break;
      work(code_b, code_a);
    }
  }

  // fold, one weight tile at a time: red[wave][m (MT*16)][n (16)]
  __syncthreads();  // the reduction area overlays the x buffers of other waves
  constexpr int kOuts = (MT * 256 + NT - 1) / NT;  // of a tile, a thread's
#pragma unroll
  for (int t = 0; t < NTL; ++t) {
    if (t < ntiles) {
      S first[kOuts];  // what the first matrix gives
#pragma unroll
      for (int mat = 0; mat < NMAT; ++mat) {
        if (t + mat > 0) __syncthreads();  // the previous tile's sums have been read
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int m = mt * 16 + 4 * kb + v;
            red[(wave * (MT * 16) + m) * 16 + r] = acc[mat * NTL + t][mt][v];
          }
        __syncthreads();
        auto output = [&](int o) {
          const int row_l = t * 16 + (o & 15);
          S res = S();
          if (row_l < rows_blk) {
            float sum = 0.f;
#pragma unroll
            for (int wv = 0; wv < NWAVES; ++wv) sum += red[wv * (MT * 256) + o];
            if (mats[mat].bias != nullptr) {
              sum += TT<T>::load(reinterpret_cast<const S*>(mats[mat].bias) + row0 + row_l);
            }
            TT<T>::store(&res, sum);
            reinterpret_cast<S*>(mats[mat].out)[(int64_t)(o >> 4) * N + row0 + row_l] = res;
          }
          return res;
        };
        if constexpr (NMAT == 1) {
          for (int o = tid; o < M * 16; o += NT) output(o);
        } else {
#pragma unroll
          for (int i = 0; i < kOuts; ++i) {
            const int o = tid + i * NT;
            if (o < M * 16) {
              const S res = output(o);
              const int row_l = t * 16 + (o & 15);
              if (mat == 0) {
                first[i] = res;
              } else if (row_l < rows_blk) {
                const float a = TT<T>::round(glu_activation(TT<T>::load(&res), act));
                TT<T>::store(reinterpret_cast<S*>(y) + (int64_t)(o >> 4) * N + row0 + row_l,
                             TT<T>::load(&first[i]) * a);
              }
            }
          }
        }
      }
    }
  }
}

template<typename T, int BITS, bool SIGNED, int ZMODE, int NWAVES, int MT, int NTL>
__global__ void __launch_bounds__(NWAVES * 64)
gemv_rows_mt(const uint16_t* __restrict__ x, const uint8_t* __restrict__ w,
             const uint16_t* __restrict__ scale, const uint16_t* __restrict__ zero,
             const uint16_t* __restrict__ bias, uint16_t* __restrict__ out, int M, int N, int K,
             int group_size, int gs_shift, int rows_per_block, int panel_chunks, int panel_groups) {
  const RowsMat mats[1] = {{w, scale, zero, bias, out}};
  gemv_rows_mt_body<T, BITS, SIGNED, ZMODE, NWAVES, MT, NTL, 1>(
      (int)blockIdx.x, x, mats, N, nullptr, 0, M, K, group_size, gs_shift, rows_per_block,
      panel_chunks, panel_groups);
}
// several linears of the same m, k and quantisation: the grid is the concatenation of their blocks
template<typename T, int BITS, bool SIGNED, int ZMODE, int NWAVES, int MT, int NTL>
__global__ void __launch_bounds__(NWAVES * 64)
gemv_rows_mt_grouped(GemvGroup g, int M, int K, int group_size, int gs_shift, int rows_per_block,
                     int panel_chunks, int panel_groups) {
  const GemvProblem pr = select_problem(g, (int)blockIdx.x);
  const RowsMat mats[1] = {{pr.w, static_cast<const uint16_t*>(pr.scale), static_cast<const uint16_t*>(pr.zero),
                            static_cast<const uint16_t*>(pr.bias), static_cast<uint16_t*>(pr.out)}};
  gemv_rows_mt_body<T, BITS, SIGNED, ZMODE, NWAVES, MT, NTL, 1>(
      (int)blockIdx.x - pr.first_block, static_cast<const uint16_t*>(pr.x), mats, pr.N, nullptr, 0, M,
      K, group_size, gs_shift, rows_per_block, panel_chunks, panel_groups);
}
template<typename T, int BITS, bool SIGNED, int ZMODE, int NWAVES, int MT, int NTL>
__global__ void __launch_bounds__(NWAVES * 64)
gemv_rows_mt_glu(const uint16_t* __restrict__ x, RowsMat hidden, RowsMat gate,
                 uint16_t* __restrict__ y, int act, int M, int N, int K, int group_size, int gs_shift,
                 int rows_per_block, int panel_chunks, int panel_groups) {
  const RowsMat mats[2] = {hidden, gate};
  gemv_rows_mt_body<T, BITS, SIGNED, ZMODE, NWAVES, MT, NTL, 2>(
      (int)blockIdx.x, x, mats, N, y, act, M, K, group_size, gs_shift, rows_per_block, panel_chunks,
      panel_groups);
}

// ---------------------------------------------------------------------------------------------
// fp32 activations (the reference registers float next to half,
// groupwise_quantization_kernels.cu:844-851): the same row split on v_mfma_f32_16x16x4_f32, one
// fp32 value of x and one of w~ per lane and MFMA.  w~ = (float(q) * s) + z, both operations
// rounded to fp32 as in the reference; products and sums are fp32 inside the matrix core.
// x (m <= 16 rows) comes from L2.
// ---------------------------------------------------------------------------------------------
template<int BITS, bool SIGNED, int ZMODE, int NWAVES>
__global__ void __launch_bounds__(NWAVES * 64)
gemv_rows_f32(const float* __restrict__ x, const uint8_t* __restrict__ w,
              const float* __restrict__ scale, const float* __restrict__ zero,
              const float* __restrict__ bias, float* __restrict__ out, int M, int N, int K,
              int group_size, int gs_shift, int rows_per_block) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int NT = NWAVES * 64;
  constexpr int CK = BITS == 4 ? 128 : 64;
  constexpr int LK = CK / 4;   // elements per lane and chunk
  constexpr int XV = LK / 4;   // 16-byte pieces of x per lane and chunk
  const int nchunks = K / CK;
  const int row_bytes = nchunks * 64;
  const int G = K / group_size;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15;
  const int kb = lane >> 4;
  const int row0 = blockIdx.x * rows_per_block;
  int rows_blk = N - row0;
  if (rows_blk > rows_per_block) rows_blk = rows_per_block;
  if (rows_blk <= 0) return;
  const int ntiles = (rows_blk + 15) >> 4;

  // LDS: [red NWAVES*256 f32][scales rows_per_block*G f32][zeros (asymmetric)]
  float* red = reinterpret_cast<float*>(smem);
  float* sl = red + NWAVES * 256;
  float* zl = sl + rows_per_block * G;

  const uint8_t* wbase = w + (int64_t)row0 * row_bytes + kb * 16;
  auto issue = [&](int tile, int c, bool live) {
    const int row_l = tile * 16 + r;
    const bool ok = row_l < rows_blk;
    const uint8_t* q = wbase + (int64_t)(ok ? row_l : 0) * row_bytes + (int64_t)c * 64;
    return __builtin_nontemporal_load(
        reinterpret_cast<const u32x4*>(live ? q : w + (int64_t)row0 * row_bytes));
  };
  int c = wave;
  u32x4 cur = issue(0, c < nchunks ? c : 0, c < nchunks);

  const int tile_elems = rows_blk * G;
  const float* stile = scale + (int64_t)row0 * G;
  const float* ztile = ZMODE == kZeroAsym ? zero + (int64_t)row0 * G : stile;
  for (int e = tid; e < tile_elems; e += NT) {
    sl[e] = stile[e];
    if (ZMODE == kZeroAsym) zl[e] = ztile[e];
  }
  __syncthreads();

  const float* xrow = x + (size_t)(r < M ? r : 0) * K + kb * LK;
  f32x4 acc[kRowsMaxTiles];
#pragma unroll
  for (int t = 0; t < kRowsMaxTiles; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  while (c < nchunks) {
    f32x4 xa[XV];
#pragma unroll
    for (int j = 0; j < XV; ++j) xa[j] = reinterpret_cast<const f32x4*>(xrow + (size_t)c * CK)[j];
    const int k0 = c * CK + kb * LK;
    const int grp = gs_shift >= 0 ? (k0 >> gs_shift) : (k0 / group_size);
#pragma unroll
    for (int t = 0; t < kRowsMaxTiles; ++t) {
      if (t < ntiles) {
        const bool last_t = t + 1 >= ntiles;
        const int nc = last_t ? c + NWAVES : c;
        const bool live = nc < nchunks;
        const u32x4 nxt = issue(last_t ? 0 : t + 1, live ? nc : 0, live);
        const int srow = (t * 16 + r) * G;
        const float s = sl[srow + grp];
        float z = 0.f;
        if (ZMODE == kZeroAsym) z = zl[srow + grp];
        if (ZMODE == kZeroSymU) z = -(float)((1 << (BITS - 1)) - 1) * s;
        // a signed container is read as offset binary; the offset leaves inside the fused
        // multiply-add (u * s - off * s is exact before its single rounding)
        const float off = SIGNED ? -(float)(1 << (BITS - 1)) * s : 0.f;
#pragma unroll
        for (int wd = 0; wd < 4; ++wd) {
          uint32_t word = cur[wd];
          if (SIGNED) word ^= (BITS == 4 ? 0x88888888u : 0x80808080u);
          if constexpr (BITS == 4) {
            const uint32_t hi = (word >> 4) & 0x0F0F0F0Fu;  // elements 0, 2, 4, 6 of the word
            const uint32_t lo = word & 0x0F0F0F0Fu;         // elements 1, 3, 5, 7
#pragma unroll
            for (int b = 0; b < 4; ++b) {
              const float u0 = (float)((hi >> (8 * b)) & 0xFFu);
              const float u1 = (float)((lo >> (8 * b)) & 0xFFu);
              float w0 = SIGNED ? __builtin_fmaf(u0, s, off) : u0 * s;
              float w1 = SIGNED ? __builtin_fmaf(u1, s, off) : u1 * s;
              if (ZMODE != kZeroNone) {
                w0 = w0 + z;
                w1 = w1 + z;
              }
              // element 8*wd + 2*b (+1) of the lane's 32: piece 2*wd + b/2 of x, component 2*(b%2)
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[2 * wd + (b >> 1)][2 * (b & 1)], w0,
                                                            acc[t], 0, 0, 0);
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[2 * wd + (b >> 1)][2 * (b & 1) + 1],
                                                            w1, acc[t], 0, 0, 0);
            }
          } else {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
              const float u0 = (float)((word >> (8 * b)) & 0xFFu);
              float w0 = SIGNED ? __builtin_fmaf(u0, s, off) : u0 * s;
              if (ZMODE != kZeroNone) w0 = w0 + z;
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[wd][b], w0, acc[t], 0, 0, 0);
            }
          }
        }
        cur = nxt;
      }
    }
    c += NWAVES;
  }

  // fold, one weight tile at a time: red[wave][m (16)][n (16)]
#pragma unroll
  for (int t = 0; t < kRowsMaxTiles; ++t) {
    if (t < ntiles) {
      if (t > 0) __syncthreads();
#pragma unroll
      for (int v = 0; v < 4; ++v) red[(wave * 16 + 4 * kb + v) * 16 + r] = acc[t][v];
      __syncthreads();
      for (int o = tid; o < M * 16; o += NT) {
        float sum = 0.f;
#pragma unroll
        for (int wv = 0; wv < NWAVES; ++wv) sum += red[wv * 256 + o];
        const int m = o >> 4;
        const int row_l = t * 16 + (o & 15);
        if (row_l < rows_blk) {
          if (bias != nullptr) sum += bias[row0 + row_l];
          out[(int64_t)m * N + row0 + row_l] = sum;
        }
      }
    }
  }
}

inline size_t gemv_rows_f32_lds_bytes(int nwaves, int K, int group_size, int rows_per_block,
                                      bool asym) {
  const int G = K / group_size;
  return (size_t)nwaves * 256 * 4 + (size_t)(asym ? 2 : 1) * rows_per_block * G * 4;
}

inline size_t gemv_rows_mt_lds_bytes(int nwaves, int mt, int bits, int rows_per_block,
                                     int panel_groups, bool asym, int matrices) {
  const size_t red = (size_t)nwaves * mt * 256 * 4;
  const size_t xb = (size_t)nwaves * mt * 16 * ((bits == 4 ? 256 : 128) + 16);
  return (xb > red ? xb : red)
         + (size_t)(matrices * (asym ? 2 : 1)) * ((rows_per_block * (panel_groups + 1) * 2 + 15) & ~15);
}

inline size_t gemv_rows_lds_bytes(int nwaves, int M, int K, int group_size, int rows_per_block,
                                  bool asym, bool staged) {
  const int G = K / group_size;
  const size_t red = (size_t)((rows_per_block + 15) / 16) * nwaves * M * 16 * 4;
  const size_t xrows = staged ? (size_t)M * (K * 2 + 16) : 0;
  return (size_t)(asym ? 2 : 1) * ((rows_per_block * G * 2 + 15) & ~15) + 64
         + (red > xrows ? red : xrows);
}

}  // namespace
}  // namespace ofq
