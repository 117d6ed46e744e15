// Streaming kernel of fused_linear_with_groupwise_quantized_weight for up to 16 rows of x, fp16 and
// bf16, 4- and 8-bit codes, groups along K from a lane's 16 bytes of codes on (32 4-bit or 16 8-bit
// elements): one linear, several in one launch, or the two of a gated linear unit with its gating.
//
// w~ = T(T(q) * s) + z with the reference's roundings
// (oneflow/user/kernels/groupwise_quantization_kernels.cu:73-117, :582-642), products and sums in fp32 in
// the matrix core, one rounding of the result.
//
// A block of 16 waves owns consecutive weight rows, cut into tiles of TR rows, and all of K.  Its waves form
// 1 .. 16 groups over the tiles and share K within a group; the host picks the split whose longest wave has
// least to do, so that the waves are busy for any row length and row count (K = 1536 gives 6 to 12 steps,
// which waves split over K alone left to 6 of 16).
//
// Everything comes by asynchronous global -> LDS copies whose completion the waves count by hand: x in natural
// order (once per block, the pieces of a record of one row and chunk XOR-swizzled), the scales of the
// block's rows (they lie together), and the codes in a ring of the wave's own, D steps of TL tiles ahead.
// Nothing is in flight in registers, nothing is converted or moved by vector instructions on the way, and
// the requests of a wave go on while it computes.
//
// Tiles.  16 rows (9 to 16 rows of x): a request of a wave is 16 rows x 64 bytes, one chunk of K, and the
// matrix instruction's 16 x 16 results are M x 16 outputs.  8 rows (up to 8 rows of x): a request is 8 rows
// x 128 bytes, lanes with bit 3 set take the next chunk; the instruction's first operand has the 8 rows of x of
// the one chunk above those of the other, so that its two diagonal 8 x 8 blocks are the partial sums of the
// two chunks (the others are nobody's) -- whole lines, no lane idle, twice as fine a split of the rows.
//
// K is any multiple of a lane's share of a chunk: in the last chunk of a ragged row the lanes beyond K
// re-read the chunk's first bytes, expand them with a scale and a zero point of 0 and meet zeros of x.
//
// The codes of 8-row tiles, whole lines, pass the caches as bytes read once: 8 x 11008 x 4096 fp16 8-bit 14.05 ->
// 13.2 us, 3 x 4096 x 4096 15.3 -> 14.5, 2 x 11008 x 4096 bf16 4-bit 23.3 -> 22.7 (weights from HBM, a zero
// point in the first and last).  Of 16-row tiles, whose requests take half a line, that made 24.2 of 23.9.
//
// What bounds it: the expansion of the codes (13 to 41 vector instructions per 8 weights) and the stream of
// them, which overlap in part, behind a fixed 4 us (launch 2.3, the first bytes, the fold and its stores).
// Taken apart at 11008 x 4096, fp16 4-bit, 8 rows of x, launches in a row: whole 10.6 us, without the codes'
// copies 8.9, without the expansion 8.7, without both 5.3, up to the first barrier 4.2.  Against gemv_rows and, for
// gated units, its grouped launch and a launch for the gating (us, 8 rows of x; more at ring_preferred):
//   bf16 4-bit   2 x 11008 x 4096  21.0 -> 17.0   2 x 4672 x 1536  10.5 -> 8.0    11008 x 4096  11.4 -> 10.8
//   fp16 8-bit   2 x 11008 x 4096  26.7 -> 24.1   2 x 4672 x 1536  11.0 -> 7.7    11008 x 4096  14.0 -> 13.5
// (zero point in the 8-bit ones).  Steps past a wave's last one that re-read it to keep the counts constant, as
// gemm_wr does, cost a memory latency at the end (0.6 us): here the counts follow the steps left.
#pragma once

#include "dequant_regs.h"
#include "gemm_kernels.h"
#include "gemv_kernels.h"
#include "gemv_rows.h"
#include "ofq_device.h"

namespace ofq {
namespace {

constexpr int kRingWaves = 16;
constexpr int kRingMaxTiles = 4;  // of a wave
template<int TL>
constexpr int ring_depth() { return TL == 1 ? 3 : (TL == 2 ? 2 : 1); }

struct RingArgs {
  int M, K, group_size, gs_shift;
  int rows_per_block;
  int wk_shift;      // 16 waves = (16 >> wk_shift) groups over the tiles x (1 << wk_shift) over K
  int phase_steps;   // steps of x in LDS at a time (all of them, or two buffers of this many)
  int phases;
  uint32_t m_magic;  // ceil(2^32 / M)
};

// bytes of LDS of the scales of one matrix
__host__ __device__ inline int ring_scale_bytes(int rows_per_block, int G) {
  return (rows_per_block * G * 2 + 16 + 15) & ~15;
}

// all but the n youngest copies have landed, n < 4
__device__ __forceinline__ void ring_wait(int n) {
  switch (n) {
    case 0: wait_vmem_all(); break;
    case 1: wait_vmem_le<1>(); break;
    case 2: wait_vmem_le<2>(); break;
    default: wait_vmem_le<3>(); break;
  }
}

// 8 fp16 values of w~ from a word of 4-bit codes in the order 1 5 0 4 3 7 2 6: a mask and an exclusive or put
// two of its nibbles behind the exponent of 1024 (low nibbles) or 64 (high ones, which stay where they are), so
// that the word takes 13 instructions (17 with a zero term) where natural order takes 20 (24).
template<bool SIGNED, int ZMODE>
__device__ __forceinline__ u32x4 dequant8_b4_f16_any_order(uint32_t word, f16x2 s2, f16x2 z2) {
  constexpr uint32_t kLo = SIGNED ? 0x64086408u : 0x64006400u, kHi = SIGNED ? 0x54805480u : 0x54005400u;
  const f16 lo = SIGNED ? (f16)-1032.0f : (f16)-1024.0f, hi = SIGNED ? (f16)-72.0f : (f16)-64.0f;
  const f16x2 lo2 = {lo, lo}, hi2 = {hi, hi};
  const uint32_t next = word >> 8;
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = i < 2 ? word : next;
    f16x2 v = (i & 1) == 0 ? __builtin_bit_cast(f16x2, (w & 0x000F000Fu) ^ kLo) + lo2
                           : __builtin_bit_cast(f16x2, (w & 0x00F000F0u) ^ kHi) + hi2;
    v = v * s2;
    if (ZMODE != kZeroNone) v = v + z2;
    o[i] = __builtin_bit_cast(uint32_t, v);
  }
  return o;
}
// x in that order
__device__ __forceinline__ u32x4 x_any_order(u32x4 v) {
  return u32x4{__builtin_amdgcn_perm(v[2], v[0], 0x07060302u), __builtin_amdgcn_perm(v[2], v[0], 0x05040100u),
               __builtin_amdgcn_perm(v[3], v[1], 0x07060302u), __builtin_amdgcn_perm(v[3], v[1], 0x05040100u)};
}

// the partial sums of one output, in order
template<int WK, int SUB>
__device__ __forceinline__ float ring_sum(const float* src, int M, int tr) {
  float part[WK][SUB];
#pragma unroll
  for (int q = 0; q < WK; ++q)
#pragma unroll
    for (int u = 0; u < SUB; ++u) part[q][u] = src[q * (M * 16) + u * (M * tr)];
  float v = 0.f;
#pragma unroll
  for (int q = 0; q < WK; ++q)
#pragma unroll
    for (int u = 0; u < SUB; ++u) v += part[q][u];
  return v;
}

template<typename T, int BITS, bool SIGNED, int ZMODE, int TR, int TL, int NMAT>
__device__ __forceinline__ void
gemv_ring_body(int block, const uint16_t* __restrict__ x, const RowsMat (&mats)[NMAT], int N,
               uint16_t* __restrict__ y, int act, const RingArgs& p) {
  typedef typename TT<T>::storage S;
  static_assert(sizeof(S) == 2, "16-bit element types");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int CK = BITS == 4 ? 128 : 64;  // elements per chunk: 64 bytes of codes per row
  constexpr int LK = CK / 4;                // elements per lane and chunk
  constexpr int XV = LK / 8;                // 16-byte pieces of x per lane and chunk
  constexpr int SUB = TR == 8 ? 2 : 1;      // chunks per step
  constexpr int kRec = CK * 2;              // bytes of x of one row and chunk
  constexpr int kPieces = kRec / 16;
  constexpr int D = ring_depth<TL>();
  constexpr bool kAnyOrder = BITS == 4 && TT<T>::dtype == OFQ_F16;
  static_assert(D * TL <= 4, "ring_wait");
  constexpr int kRegions = ZMODE == kZeroAsym ? 2 : 1;
  const int M = p.M, K = p.K;
  const int row_bytes = K / LK * 16;
  const int G = p.gs_shift >= 0 ? K >> p.gs_shift : K / p.group_size;
  const int steps = (K + CK * SUB - 1) / (CK * SUB);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int WK = 1 << p.wk_shift;
  const int wk = wave & (WK - 1), wt = wave >> p.wk_shift;
  const int r = lane & 15;
  const int kb = lane >> 4;
  const int trow = r & (TR - 1);                // row of the tile
  const int sub = SUB == 2 ? r >> 3 : 0;        // chunk of the step
  const int row0 = block * p.rows_per_block;
  int rows_blk = N - row0;
  if (rows_blk > p.rows_per_block) rows_blk = p.rows_per_block;
  if (rows_blk <= 0) return;
  const int ntiles = (rows_blk + TR - 1) / TR;  // per matrix
  const int nvt = NMAT * ntiles;

  // LDS: [scales, zeros of every matrix][rings of the waves][x, one or two buffers]; the sums take
  //      the place of all of it
  const int sreg = ring_scale_bytes(p.rows_per_block, G);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const int ring0 = ((NMAT * kRegions * sreg + 1023) & ~1023) + wave * (D * TL * 1024);
  const int xbase = ((NMAT * kRegions * sreg + 1023) & ~1023) + kRingWaves * (D * TL * 1024);
  const int xbuf_bytes = (p.phase_steps * SUB * M * kRec + 1023) & ~1023;

  // the last 16-byte piece of the scales may straddle the end of the array: of the blocks whose rows reach
  // into it element by element, and first (a load that the compiler waits for waits for the copies before it
  // as well)
  const int64_t all_bytes = (int64_t)N * G * 2;
  const int64_t s_first = (int64_t)row0 * G * 2;
  const int s_shift = (int)(s_first & 15);
  const int s_bytes = s_shift + rows_blk * G * 2;
  const int64_t s_end = s_first + (int64_t)rows_blk * G * 2;
  if (s_end > (all_bytes & ~(int64_t)15)) {
    const int64_t e = (all_bytes >> 4) * 8 + tid;
    if (tid < 8 && e * 2 < s_end && e * 2 >= s_first) {
#pragma unroll
      for (int mt = 0; mt < NMAT; ++mt) {
        uint8_t* at = smem + mt * kRegions * sreg + (e * 2 - s_first) + s_shift;
        *reinterpret_cast<uint16_t*>(at) = mats[mt].scale[e];
        if (ZMODE == kZeroAsym) *reinterpret_cast<uint16_t*>(at + sreg) = mats[mt].zero[e];
      }
    }
  }

  // bias of the first output that this thread adds up at the end
  const int padded = ntiles * TR;
  uint16_t bias_raw[NMAT] = {};
  if (tid < M * padded) {
    const int row_l = tid % padded;
#pragma unroll
    for (int mt = 0; mt < NMAT; ++mt)
      if (mats[mt].bias != nullptr && row_l < rows_blk) bias_raw[mt] = mats[mt].bias[row0 + row_l];
  }

  // ---- copies -----------------------------------------------------------------------------------
  auto swizzle = [&](int m, int odd) {
    if constexpr (BITS == 4) return SUB == 2 ? m | (odd << 3) : m;
    else return SUB == 2 ? (m >> 1) | (odd << 2) : m >> 1;
  };
  auto copy_x = [&](int phase) {
    const int buf = xbase + (phase & 1) * xbuf_bytes;
    const int c0 = phase * p.phase_steps * SUB;
    const int left = steps * SUB - c0;
    const int nrec = (left < p.phase_steps * SUB ? left : p.phase_steps * SUB) * M;
    const int nops = (nrec * kRec + 1023) >> 10;
    for (int op = wave; op < nops; op += kRingWaves) {
      const int rec = op * (1024 / kRec) + lane / kPieces;
      const int c = (int)__umulhi((uint32_t)rec, p.m_magic);
      const int m = M == 1 ? 0 : rec - c * M;
      const int cl = M == 1 ? rec : c;
      const int piece = (lane % kPieces) ^ swizzle(m, cl & 1);
      const int byte = (c0 + cl) * kRec + piece * 16;
      if (rec < nrec && byte < K * 2) {
        async_copy16_at(reinterpret_cast<const uint8_t*>(x), (uint32_t)(m * K * 2 + byte),
                        lds0 + buf + op * 1024);
      } else {
        *reinterpret_cast<u32x4*>(smem + buf + op * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
      }
    }
  };
  auto copy_scales = [&]() {
#pragma unroll
    for (int i = 0; i < NMAT * kRegions; ++i) {
      const RowsMat& mt = mats[i / kRegions];
      const uint8_t* src = reinterpret_cast<const uint8_t*>(i % kRegions == 0 ? mt.scale : mt.zero)
                           + (s_first - s_shift);
      const int nops = (s_bytes + 1023) >> 10;
      for (int op = wave; op < nops; op += kRingWaves) {
        const int o = op * 1024 + lane * 16;
        if (o < s_bytes && s_first - s_shift + o + 16 <= all_bytes) {
          async_copy16_at(src, (uint32_t)o, lds0 + i * sreg + op * 1024);
        }
      }
    }
  };
  uint32_t roff[TL];         // of this lane's row of every tile, and its place in a step
  const uint8_t* wbase[TL];  // (the same for every lane)
  int srow[TL];              // LDS bytes of its scales
#pragma unroll
  for (int t = 0; t < TL; ++t) {
    const int vt = wt * TL + t;
    const bool second = NMAT == 2 && vt >= ntiles;
    const int row_l = (second ? vt - ntiles : vt) * TR + trow;
    const bool ok = vt < nvt && row_l < rows_blk;
    roff[t] = (ok ? (uint32_t)row_l * (uint32_t)row_bytes : 0u) + (uint32_t)(sub * 64 + kb * 16);
    wbase[t] = mats[NMAT == 2 && second ? NMAT - 1 : 0].w + (int64_t)row0 * row_bytes;
    srow[t] = (second ? kRegions * sreg : 0) + s_shift + (ok ? row_l : 0) * G * 2;
  }
  // codes of a step's tile; bytes past the row's end re-read the step's first ones
  auto copy_codes = [&](int s, int slot, int t) {
    const uint32_t at = (uint32_t)s * (SUB * 64u);
    uint32_t off = roff[t];
    if ((int)at + SUB * 64 > row_bytes) {  // (the same for every lane)
      if ((int)at + sub * 64 + kb * 16 >= row_bytes) off -= (uint32_t)(sub * 64 + kb * 16);
    }
    const uint32_t to = lds0 + ring0 + (slot * TL + t) * 1024;
    if constexpr (SUB == 2) async_copy16_once(wbase[t] + at, off, to);
    else async_copy16_at(wbase[t] + at, off, to);
  };
  // of this wave's steps from s on, how many are among the next n
  auto live_steps = [&](int s, int n) {
    int live = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) live += d < n && s + d * WK < steps ? 1 : 0;
    return live;
  };
  copy_x(0);
  copy_scales();
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (wk + d * WK < steps) {
#pragma unroll
      for (int t = 0; t < TL; ++t) copy_codes(wk + d * WK, d, t);
    }

  f32x4 acc[TL][2];
#pragma unroll
  for (int t = 0; t < TL; ++t) {
    acc[t][0] = f32x4{0.f, 0.f, 0.f, 0.f};
    acc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // this lane's pieces of x within a step: row r of x (rows >= M repeat the last one and feed results that
  // are nobody's)
  int xoff[XV];
  {
    const int m = trow < M ? trow : M - 1;
    const int key = swizzle(m, sub);
#pragma unroll
    for (int j = 0; j < XV; ++j) xoff[j] = (sub * M + m) * kRec + (((kb * XV + j) ^ key) << 4);
  }
  // x, scales and zeros have landed, everyone's; the codes stay in flight
  switch (live_steps(wk, D)) {
    case 0: wait_vmem_all(); break;
    case 1: wait_vmem_le<TL>(); break;
    case 2: wait_vmem_le<2 * TL>(); break;
    default: wait_vmem_le<3 * TL>(); break;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  int s = wk, slot = 0;
  for (int phase = 0; phase < p.phases; ++phase) {
    if (phase + 1 < p.phases) copy_x(phase + 1);  // (its buffer's last readers have passed a barrier)
    const int first = phase * p.phase_steps;
    const int last = steps < first + p.phase_steps ? steps : first + p.phase_steps;
    const uint8_t* xb = smem + xbase + (phase & 1) * xbuf_bytes;
    int newer = 0;  // steps requested behind the next phase's x
    for (; s < last; s += WK) {
      const uint8_t* xp = xb + (s - first) * (SUB * M * kRec);
      u32x4 xa[XV];
#pragma unroll
      for (int j = 0; j < XV; ++j) xa[j] = *reinterpret_cast<const u32x4*>(xp + xoff[j]);
      if (kAnyOrder) {
#pragma unroll
        for (int j = 0; j < XV; ++j) xa[j] = x_any_order(xa[j]);
      }
      int k0 = (s * SUB + sub) * CK + kb * LK;
      const bool in_row = k0 < K;
      k0 = in_row ? k0 : 0;
      const int grp = p.gs_shift >= 0 ? (k0 >> p.gs_shift) : (k0 / p.group_size);
      const bool more = s + D * WK < steps;
      const int younger = live_steps(s + WK, D - 1) * TL + TL - 1;
      const uint8_t* cp = smem + ring0 + slot * (TL * 1024) + lane * 16;
#pragma unroll
      for (int t = 0; t < TL; ++t) {
        // younger than this tile's copy: those of later steps, of the step's later tiles, and, if there
        // is such a step, what has taken the slots of its earlier tiles
        ring_wait(more ? younger : younger - t);
        asm volatile("" ::: "memory");
        const u32x4 codes = *reinterpret_cast<const u32x4*>(cp + t * 1024);
        const uint16_t sraw = *reinterpret_cast<const uint16_t*>(smem + srow[t] + grp * 2);
        uint16_t zraw = 0;
        if (ZMODE == kZeroAsym) zraw = *reinterpret_cast<const uint16_t*>(smem + srow[t] + sreg + grp * 2);
        // the codes are in registers: their slot is free
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (more) copy_codes(s + D * WK, slot, t);
        if (wt * TL + t < nvt) {
          const float sc = in_row ? raw16_to_float<T>(sraw) : 0.f;
          float z = 0.f;
          if (ZMODE == kZeroAsym) z = in_row ? raw16_to_float<T>(zraw) : 0.f;
          if (ZMODE == kZeroSymU) z = TT<T>::round(-(float)((1 << (BITS - 1)) - 1) * sc);
          if constexpr (BITS == 4) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              u32x4 b;
              if constexpr (kAnyOrder) {
                const f16x2 s2 = {(f16)sc, (f16)sc}, z2 = {(f16)z, (f16)z};  // (exact)
                b = dequant8_b4_f16_any_order<SIGNED, ZMODE>(codes[j], s2, z2);
              } else {
                b = dequant8_b4<T, SIGNED, ZMODE>(codes[j], sc, z);
              }
              // two accumulators: consecutive matrix instructions do not wait for each other
              acc[t][j & 1] = MfmaK32<T>::mma(xa[j], b, acc[t][j & 1]);
            }
          } else {
            u32x4 b0, b1;
            dequant16_b8<T, SIGNED, ZMODE>(codes, sc, z, b0, b1);
            acc[t][0] = MfmaK32<T>::mma(xa[0], b0, acc[t][0]);
            acc[t][1] = MfmaK32<T>::mma(xa[1], b1, acc[t][1]);
          }
        }
      }
      newer += more ? 1 : 0;
      slot = slot + 1 == D ? 0 : slot + 1;
    }
    if (phase + 1 < p.phases) {
      const int flying = live_steps(s, D);
      const int younger = newer < flying ? newer : flying;
      ring_wait(younger * TL < 4 ? younger * TL : 3);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
  }

  // ---- sums of the waves -> LDS, [tile][wave of K][chunk of the step][M][TR] ------------------------
  __syncthreads();
  float* red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int t = 0; t < TL; ++t) {
    const int vt = wt * TL + t;
    if (vt < nvt) {
      float* dst = red + (size_t)((vt << p.wk_shift) + wk) * (M * 16);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 4 * kb + v;  // row of the result
        const int m = i & (TR - 1);
        if (m < M && (SUB == 1 || (i >> 3) == sub)) {
          dst[(SUB == 2 ? sub * M + m : m) * TR + trow] = acc[t][0][v] + acc[t][1][v];
        }
      }
    }
  }
  __syncthreads();
  for (int o = tid; o < M * padded; o += kRingWaves * 64) {
    const int m = o / padded;
    const int row_l = o - m * padded;
    const int tile = row_l / TR;
    float sum[NMAT];
#pragma unroll
    for (int mt = 0; mt < NMAT; ++mt) {
      const float* src = red + (size_t)((mt * ntiles + tile) << p.wk_shift) * (M * 16) + m * TR
                         + (row_l & (TR - 1));
      float v;
      switch (p.wk_shift) {  // (unrolled: the reads of a sum go out together)
        case 4: v = ring_sum<16, SUB>(src, M, TR); break;
        case 3: v = ring_sum<8, SUB>(src, M, TR); break;
        case 2: v = ring_sum<4, SUB>(src, M, TR); break;
        case 1: v = ring_sum<2, SUB>(src, M, TR); break;
        default: v = ring_sum<1, SUB>(src, M, TR); break;
      }
      sum[mt] = v;
    }
    if (row_l < rows_blk) {
      const int64_t at = (int64_t)m * N + row0 + row_l;
      S res[NMAT];
#pragma unroll
      for (int mt = 0; mt < NMAT; ++mt) {
        float v = sum[mt];
        if (o == tid) {
          v += raw16_at_end<T>(bias_raw[mt]);
        } else if (mats[mt].bias != nullptr) {
          v += TT<T>::load(reinterpret_cast<const S*>(mats[mt].bias) + row0 + row_l);
        }
        TT<T>::store(&res[mt], v);
        reinterpret_cast<S*>(mats[mt].out)[at] = res[mt];
      }
      if constexpr (NMAT == 2) {
        const float a = TT<T>::round(glu_activation(TT<T>::load(&res[1]), act));
        TT<T>::store(reinterpret_cast<S*>(y) + at, TT<T>::load(&res[0]) * a);
      }
    }
  }
}

template<typename T, int BITS, bool SIGNED, int ZMODE, int TR, int TL>
__global__ void __launch_bounds__(kRingWaves * 64)
gemv_ring(const uint16_t* __restrict__ x, RowsMat mat, int N, RingArgs p) {
  const RowsMat mats[1] = {mat};
  gemv_ring_body<T, BITS, SIGNED, ZMODE, TR, TL, 1>((int)blockIdx.x, x, mats, N, nullptr, 0, p);
}
// Several linears of the same m, k and quantisation: the grid is the concatenation of their blocks.
template<typename T, int BITS, bool SIGNED, int ZMODE, int TR, int TL>
__global__ void __launch_bounds__(kRingWaves * 64)
gemv_ring_grouped(GemvGroup g, RingArgs p) {
  const GemvProblem pr = select_problem(g, (int)blockIdx.x);
  const RowsMat mats[1] = {{pr.w, static_cast<const uint16_t*>(pr.scale), static_cast<const uint16_t*>(pr.zero),
                            static_cast<const uint16_t*>(pr.bias), static_cast<uint16_t*>(pr.out)}};
  gemv_ring_body<T, BITS, SIGNED, ZMODE, TR, TL, 1>((int)blockIdx.x - pr.first_block,
                                                    static_cast<const uint16_t*>(pr.x), mats, pr.N,
                                                    nullptr, 0, p);
}
// hidden = x w^T + b -> out, gate = x v^T + c -> out2, y = hidden * act(gate): a block owns the same rows
// of both weights.
template<typename T, int BITS, bool SIGNED, int ZMODE, int TR, int TL>
__global__ void __launch_bounds__(kRingWaves * 64)
gemv_ring_glu(const uint16_t* __restrict__ x, RowsMat hidden, RowsMat gate, int N,
              uint16_t* __restrict__ y, int act, RingArgs p) {
  const RowsMat mats[2] = {hidden, gate};
  gemv_ring_body<T, BITS, SIGNED, ZMODE, TR, TL, 2>((int)blockIdx.x, x, mats, N, y, act, p);
}

}  // namespace
}  // namespace ofq
