// Streaming kernel of fused_linear_with_groupwise_quantized_weight for up to 48 rows of x whose waves share
// nothing but scales: fp16 and bf16, 4- and 8-bit codes, groups along K from a lane's 16 bytes of codes on; one linear,
// several in one launch, or the two of a gated linear unit with its gating.
//
// w~ = T(T(q) * s) + z with the reference's roundings
// (oneflow/user/kernels/groupwise_quantization_kernels.cu:73-117, :582-642), products and sums in fp32 in
// the matrix core, one rounding of the result; up to 16 rows of x, symmetric 4-bit
// fp16 codes in groups of whole chunks meet x as they are and their scale multiplies the chunk's fp32 sum (LATE: closer
// to exact arithmetic than the rounded w~, and what gemv_w4p_f16 does with them).
//
// A block owns consecutive weight rows, walked as TL 16-row tiles, and all of K.  A wave takes every NW-th step of
// 128 bytes of codes (two chunks of K; above 16 rows of x with 4-bit codes 64), and both its columns of x and the codes of all tiles come by
// asynchronous global -> LDS copies to a place of its own: no wave waits for another between
// the scales, which the block copies once, and the sums at the end.  Copies take whole lines (8 rows x 128 bytes of codes;
// 256 or 512 bytes of a row of x), their pieces XOR-swizzled on the way so that operand reads meet no conflict of
// banks.  The next step's x and tiles are requested one by one, as the present ones have been read into registers.
//
// What bounds it: the expansion of the codes and the stream of them, two waves a SIMD, behind about 2.5 us of launch,
// first bytes and sums.  8 x 4096 x 11008 fp16 4-bit in groups of 128 takes 8.7 us (x, copied by all waves behind a
// barrier in two parts, made it 11.0 in gemv_w4p_f16), 16 rows 10.7 (13.5); 8 rows of x of 3 x 4096 x 4096 fp16 4-bit in groups of 128 take 9.0 us (10.8 in
// gemv_w4p_f16_grouped), 16 of 2 x 11008 x 4096 13.0 (23.5); weights from HBM.  A step in LDS and not two or three: with more in flight from the start
// every wave's first step comes later (8 x 4096 x 11008 10.7 us).  Above 16 rows x and codes come in at 45 to 55 bytes
// per ns and CU together: 48 x 11008 x 4096 with a zero point 15.8 us, 64 rows 17.4 and more (not taken).  Codes of a tile read before the products of the tile
// ahead of it: 1 to 2 %; offsets of copies formed once: 2 to 5 %.  What else it is measured against: gemv_flow_choice.
//
// K is any multiple of a lane's share of a chunk: lanes beyond K re-read a step's first bytes, and take x, scale and zero
// point as 0.
#pragma once

#include "dequant_regs.h"
#include "gemm_kernels.h"
#include "gemv_kernels.h"
#include "gemv_ring.h"
#include "gemv_rows.h"
#include "ofq_device.h"

namespace ofq {
namespace {

struct FlowArgs {
  int M, K, group_size, gs_shift;
  int rows_per_block;
};

// 8 4-bit codes, two's complement, as they are behind the exponents of 1024 (low nibbles: 1032 + q) and 64 (high
// nibbles, which stay where they are: 72 + q), in the order 1 5 0 4 3 7 2 6; 5 instructions a word, all exact.  What
// is added to the codes meets x as well and is taken off per chunk.
__device__ __forceinline__ u32x4 biased8_b4_f16_any_order(uint32_t word) {
  const uint32_t next = word >> 8;
  return u32x4{(word & 0x000F000Fu) ^ 0x64086408u, (word & 0x00F000F0u) ^ 0x54805480u,
               (next & 0x000F000Fu) ^ 0x64086408u, (next & 0x00F000F0u) ^ 0x54805480u};
}

// Chunks of K in a step, MX eights of rows of x: two, whole lines of the codes, or where a step's x would leave no
// room for as many waves, one (a line's halves are then those of neighbouring waves).
__host__ __device__ constexpr int flow_chunks(int bits, int mx) { return bits == 4 && mx > 2 ? 1 : 2; }
// 1 KB copies of x in a step, and of a tile's codes
__host__ __device__ constexpr int flow_x_ops(int bits, int mx) { return mx * flow_chunks(bits, mx) * (bits == 4 ? 2 : 1); }
template<int I>
struct FlowConst { static constexpr int value = I; };
template<int I, int N, typename F>
__device__ __forceinline__ void flow_for(F&& f) {
  if constexpr (I < N) {
    f(FlowConst<I>());
    flow_for<I + 1, N>(f);
  }
}

template<typename T, int BITS, bool SIGNED, int ZMODE, bool LATE, bool TILED, int MX, int TL, int NMAT, int NW>
__device__ __forceinline__ void
gemv_flow_body(int block, const uint16_t* __restrict__ x, const RowsMat (&mats)[NMAT], int N,
               uint16_t* __restrict__ y, int act, const FlowArgs& p) {
  typedef typename TT<T>::storage S;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int CK = BITS == 4 ? 128 : 64;  // elements per chunk: 64 bytes of codes per row
  constexpr int LK = CK / 4;                // elements per lane and chunk
  constexpr int XV = LK / 8;                // 16-byte pieces of x per lane and chunk
  constexpr int NT = TL * NMAT;             // tiles
  constexpr int CH = flow_chunks(BITS, MX); // chunks per step, and copies of a tile
  constexpr int MT = (MX + 1) / 2;          // 16-row tiles of x
  constexpr int kXRow = CK * 2 * CH;        // bytes of x of one row and step
  constexpr int kXPieces = kXRow / 16;
  constexpr int kXOps = flow_x_ops(BITS, MX);
  constexpr int STEP = kXOps + CH * NT;     // copies of a step, 1 KB each: x, then tile by tile
  constexpr int kStepBytes = CH * 64;       // of codes of one row
  constexpr int kSums = MT == 1 ? 2 : 1;    // of a tile: consecutive matrix instructions do not wait for each other
  static_assert(MT == 1 || CH == 1 || BITS == 8, "one sum for two chunks");
  constexpr bool kAnyOrder = BITS == 4 && TT<T>::dtype == OFQ_F16;
  constexpr int kRegions = ZMODE == kZeroAsym ? 2 : 1;
  static_assert(2 * STEP < 63, "vmcnt is a 6-bit counter");
  static_assert(!TILED || (CH == 2 && NMAT == 1 && BITS == 4), "a tile-major copy has 1 KB per tile and chunk");
  static_assert(!LATE || (kAnyOrder && SIGNED && ZMODE == kZeroNone), "one scale a chunk and nothing to add");
  const int M = p.M, K = p.K;
  const int row_bytes = K / LK * 16;
  const int G = p.gs_shift >= 0 ? K >> p.gs_shift : K / p.group_size;
  const int steps = (K + CH * CK - 1) / (CH * CK);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15;
  const int kb = lane >> 4;
  const int row0 = block * p.rows_per_block;
  int rows_blk = N - row0;
  if (rows_blk > p.rows_per_block) rows_blk = p.rows_per_block;
  if (rows_blk <= 0) return;

  // LDS: [scales, zeros of every matrix][rings of the waves]; the sums take the place of all of it
  const int sreg = ring_scale_bytes(p.rows_per_block, G);
  const int ring0 = ((NMAT * kRegions * sreg + 1023) & ~1023) + wave * (STEP * 1024);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;

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
  // the bias of a thread's outputs, all of one row, without a branch and before the copies
  constexpr int R = TL * 16;
  const int orow = tid % R;
  uint16_t bias_raw[NMAT];
#pragma unroll
  for (int mt = 0; mt < NMAT; ++mt) {
    const uint16_t* at = mats[mt].bias != nullptr ? mats[mt].bias + row0 : mats[mt].scale + s_first / 2;
    bias_raw[mt] = at[orow < rows_blk ? orow : 0];
  }

  // ---- copies -----------------------------------------------------------------------------------
#pragma unroll
  for (int i = 0; i < NMAT * kRegions; ++i) {
    const RowsMat& mt = mats[i / kRegions];
    const uint8_t* src = reinterpret_cast<const uint8_t*>(i % kRegions == 0 ? mt.scale : mt.zero) + (s_first - s_shift);
    const int nops = (s_bytes + 1023) >> 10;
    for (int op = wave; op < nops; op += NW) {
      const int o = op * 1024 + lane * 16;
      if (o < s_bytes && s_first - s_shift + o + 16 <= all_bytes) {
        async_copy16_at(src, (uint32_t)o, lds0 + i * sreg + op * 1024);
      }
    }
  }
  // x: 1024 / kXRow rows a copy; rows >= M re-read the last one and feed results that are nobody's
  // (offsets within a whole step; the one that K ends in keeps its lanes in the row by its own)
  uint32_t xoff[kXOps];
  auto x_piece = [&](int o) { return (uint32_t)(((lane % kXPieces) ^ ((o * (1024 / kXRow) + lane / kXPieces) & 15)) << 4); };
#pragma unroll
  for (int o = 0; o < kXOps; ++o) {
    const int row = o * (1024 / kXRow) + lane / kXPieces;
    xoff[o] = (uint32_t)(row < M ? row : M - 1) * (uint32_t)(K * 2) + x_piece(o);
  }
  auto copy_x = [&](int s) {
    const uint8_t* base = reinterpret_cast<const uint8_t*>(x) + (int64_t)s * kXRow;
    if ((s + 1) * kXRow <= K * 2) {
#pragma unroll
      for (int o = 0; o < kXOps; ++o) async_copy16_at(base, xoff[o], lds0 + ring0 + o * 1024);
    } else {
#pragma unroll
      for (int o = 0; o < kXOps; ++o) {
        const uint32_t piece = x_piece(o);
        async_copy16_at(base, s * kXRow + (int)piece < K * 2 ? xoff[o] : xoff[o] - piece, lds0 + ring0 + o * 1024);
      }
    }
  };
  // codes: two eights a tile, or 16 rows of half a line
  uint32_t woff[TL][CH], wpiece[CH];
#pragma unroll
  for (int h = 0; h < CH; ++h) {
    const int row = CH == 2 ? h * 8 + (lane >> 3) : lane >> 2;
    wpiece[h] = (uint32_t)((CH == 2 ? (lane & 7) ^ (row >> 1) : (lane & 3) ^ (row >> 2)) << 4);
#pragma unroll
    for (int t = 0; t < TL; ++t) {
      woff[t][h] = (uint32_t)(t * 16 + row < rows_blk ? t * 16 + row : rows_blk - 1) * (uint32_t)row_bytes + wpiece[h];
    }
  }
  const uint8_t* wbase[NMAT];
#pragma unroll
  for (int mt = 0; mt < NMAT; ++mt) wbase[mt] = mats[mt].w + (int64_t)row0 * row_bytes;
  auto copy_codes = [&](const uint8_t* base, uint32_t off, uint32_t to) {
    if constexpr (CH == 2) async_copy16_once(base, off, to);
    else async_copy16_at(base, off, to);
  };
  auto copy_tile = [&](int s, int t) {
    if constexpr (TILED) {
      const int chunks = K / CK;
      const uint8_t* base = mats[0].w + (((int64_t)block * TL + t) * chunks + s * CH) * 1024;
#pragma unroll
      for (int h = 0; h < CH; ++h) {
        copy_codes(base, (s * CH + h < chunks ? h * 1024u : 0u) + lane * 16u, lds0 + ring0 + (kXOps + CH * t + h) * 1024);
      }
      return;
    }
    const uint8_t* base = wbase[t / TL] + (int64_t)s * kStepBytes;
    const uint32_t to = lds0 + ring0 + (kXOps + CH * t) * 1024;
    if ((s + 1) * kStepBytes <= row_bytes) {
#pragma unroll
      for (int h = 0; h < CH; ++h) copy_codes(base, woff[t % TL][h], to + h * 1024);
    } else {
#pragma unroll
      for (int h = 0; h < CH; ++h) {
        copy_codes(base, woff[t % TL][h] - (s * kStepBytes + (int)wpiece[h] < row_bytes ? 0u : wpiece[h]), to + h * 1024);
      }
    }
  };
  if (wave < steps) {
    copy_x(wave);
#pragma unroll
    for (int t = 0; t < NT; ++t) copy_tile(wave, t);
  }
  // scales and zeros have landed, everyone's; the rest stays in flight
  if (wave < steps) wait_vmem_le<STEP>();
  else wait_vmem_all();
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // ---- products ---------------------------------------------------------------------------------
  f32x4 acc[NT][MT][kSums];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < kSums; ++i) acc[t][mt][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  int xat[CH][XV];  // this lane's pieces of x in a step, of row r of a tile (of a tile of one eight: its rows twice)
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int j = 0; j < XV; ++j) {
      const int row = MX == 1 ? r & 7 : r;
      xat[c][j] = row * kXRow + (((c * 4 + kb) * XV + j) ^ row) * 16;
    }
  int cat[CH];      // and of a tile's codes
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    if constexpr (TILED) cat[c] = c * 1024 + lane * 16;  // (as the copy has them)
    else cat[c] = CH == 2 ? r * 128 + (((c * 4 + kb) ^ (r >> 1)) << 4) : r * 64 + ((kb ^ (r >> 2)) << 4);
  }
  int srow[TL];
#pragma unroll
  for (int t = 0; t < TL; ++t) srow[t] = s_shift + (t * 16 + r < rows_blk ? t * 16 + r : rows_blk - 1) * G * 2;

  for (int s = wave; s < steps; s += NW) {
    const bool more = s + NW < steps;
    wait_vmem_le<CH * NT>();
    asm volatile("" ::: "memory");
    u32x4 xa[CH][MT][XV];
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < XV; ++j)
          xa[c][mt][j] = *reinterpret_cast<const u32x4*>(smem + ring0 + mt * (16 * kXRow) + xat[c][j]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) copy_x(s + NW);
    bool in_row[CH];
    int grp[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      int k0 = (s * CH + c) * CK + kb * LK;
      in_row[c] = k0 < K;
      k0 = in_row[c] ? k0 : 0;
      grp[c] = (p.gs_shift >= 0 ? k0 >> p.gs_shift : k0 / p.group_size) * 2;
    }
    if ((s + 1) * CH * CK > K) {
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int j = 0; j < XV; ++j)
            if (!in_row[c]) xa[c][mt][j] = u32x4{0u, 0u, 0u, 0u};
    }
    if constexpr (kAnyOrder) {
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int j = 0; j < XV; ++j) xa[c][mt][j] = x_any_order(xa[c][mt][j]);
    }
    // minus what the exponents add to the codes' values, of every row of x
    f32x4 corr[CH][MT];
    if constexpr (LATE) {
      uint32_t lo = 0xE408E408u, hi = 0xD480D480u;  // (-1032, -1032), (-72, -72)
      asm volatile("" : "+v"(lo), "+v"(hi));
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          corr[c][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int j = 0; j < XV; ++j) corr[c][mt] = MfmaK32<T>::mma(xa[c][mt][j], u32x4{lo, hi, lo, hi}, corr[c][mt]);
        }
    }
    // a tile's codes are read while the products of the one before it are under way
    u32x4 codes[CH];
    uint16_t sraw[CH], zraw[CH] = {};
    auto read_tile = [&](auto index) {
      constexpr int t = decltype(index)::value;
      // younger than its copies: those of the tiles after it and, if there is a next step, its x and tiles before t
      if (more) wait_vmem_le<CH * (NT - 1) + kXOps>();
      else wait_vmem_le<CH * (NT - 1 - t)>();
      asm volatile("" ::: "memory");
      const uint8_t* cp = smem + ring0 + (kXOps + CH * t) * 1024;
      const uint8_t* sp = smem + (t / TL) * kRegions * sreg + srow[t % TL];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        codes[c] = *reinterpret_cast<const u32x4*>(cp + cat[c]);
        sraw[c] = *reinterpret_cast<const uint16_t*>(sp + grp[c]);
        if (ZMODE == kZeroAsym) zraw[c] = *reinterpret_cast<const uint16_t*>(sp + sreg + grp[c]);
      }
    };
    read_tile(FlowConst<0>());
    flow_for<0, NT>([&](auto index) {
      constexpr int t = decltype(index)::value;
      // the codes are in registers: their place is free
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (more) copy_tile(s + NW, t);
      u32x4 q[CH];
      float sc[CH], z[CH];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        q[c] = codes[c];
        sc[c] = in_row[c] ? raw16_to_float<T>(sraw[c]) : 0.f;
        z[c] = 0.f;
        if (ZMODE == kZeroAsym) z[c] = in_row[c] ? raw16_to_float<T>(zraw[c]) : 0.f;
        if (ZMODE == kZeroSymU) z[c] = TT<T>::round(-(float)((1 << (BITS - 1)) - 1) * sc[c]);
      }
      if constexpr (t + 1 < NT) read_tile(FlowConst<t + 1>());
      if constexpr (LATE) {
        f32x4 sum[CH][MT];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int c = 0; c < CH; ++c) {
            const u32x4 b = biased8_b4_f16_any_order(q[c][j]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
              sum[c][mt] = MfmaK32<T>::mma(xa[c][mt][j], b, j == 0 ? corr[c][mt] : sum[c][mt]);
          }
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              acc[t][mt][c % kSums][v] = __builtin_fmaf(sum[c][mt][v], sc[c], acc[t][mt][c % kSums][v]);
      } else if constexpr (BITS == 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int c = 0; c < CH; ++c) {
            u32x4 b;
            if constexpr (kAnyOrder) {
              const f16x2 s2 = {(f16)sc[c], (f16)sc[c]}, z2 = {(f16)z[c], (f16)z[c]};  // (exact)
              b = dequant8_b4_f16_any_order<SIGNED, ZMODE>(q[c][j], s2, z2);
            } else {
              b = dequant8_b4<T, SIGNED, ZMODE>(q[c][j], sc[c], z[c]);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
              acc[t][mt][c % kSums] = MfmaK32<T>::mma(xa[c][mt][j], b, acc[t][mt][c % kSums]);
          }
      } else {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          u32x4 b0, b1;
          dequant16_b8<T, SIGNED, ZMODE>(q[c], sc[c], z[c], b0, b1);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[t][mt][c % kSums] = MfmaK32<T>::mma(xa[c][mt][0], b0, acc[t][mt][c % kSums]);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[t][mt][c % kSums] = MfmaK32<T>::mma(xa[c][mt][1], b1, acc[t][mt][c % kSums]);
        }
      }
    });
  }

  // ---- sums of the waves, [wave][row of x][row of w + 4] ------------------------------------------------
  __syncthreads();
  float* red = reinterpret_cast<float*>(smem);
  constexpr int RP = NT * 16 + 4;
  const int waves = steps < NW ? steps : NW;  // that have a sum
  if (wave < waves) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = mt * 16 + 4 * kb + v;
        if (m < M) {
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            float sum = acc[t][mt][0][v];
            if constexpr (kSums == 2) sum += acc[t][mt][1][v];
            red[(wave * M + m) * RP + t * 16 + r] = sum;
          }
        }
      }
  }
  __syncthreads();
  constexpr int kRowsAtOnce = NW * 64 / R;
  if (tid >= kRowsAtOnce * R || orow >= rows_blk) return;
  float bias[NMAT];
#pragma unroll
  for (int mt = 0; mt < NMAT; ++mt) bias[mt] = mats[mt].bias != nullptr ? raw16_at_end<T>(bias_raw[mt]) : 0.f;
  for (int m = tid / R; m < M; m += kRowsAtOnce) {
    const int64_t at = (int64_t)m * N + row0 + orow;
    S res[NMAT];
#pragma unroll
    for (int mt = 0; mt < NMAT; ++mt) {
      const float* src = red + m * RP + mt * R + orow;
      float v = 0.f;
      if (waves == NW) {
        float part[NW];
#pragma unroll
        for (int w = 0; w < NW; ++w) part[w] = src[w * M * RP];
#pragma unroll
        for (int w = 0; w < NW; ++w) v += part[w];
      } else {
        for (int w = 0; w < waves; ++w) v += src[w * M * RP];
      }
      if (mats[mt].bias != nullptr) v += bias[mt];
      TT<T>::store(&res[mt], v);
      reinterpret_cast<S*>(mats[mt].out)[at] = res[mt];
    }
    if constexpr (NMAT == 2) {
      const float a = TT<T>::round(glu_activation(TT<T>::load(&res[1]), act));
      TT<T>::store(reinterpret_cast<S*>(y) + at, TT<T>::load(&res[0]) * a);
    }
  }
}

// TILED: the codes as the tile-major copy of the weight has them, rows_per_block of its split.
template<typename T, int BITS, bool SIGNED, int ZMODE, bool LATE, bool TILED, int MX, int TL, int NW>
__global__ void __launch_bounds__(NW * 64)
gemv_flow(const uint16_t* __restrict__ x, RowsMat mat, int N, FlowArgs p) {
  const RowsMat mats[1] = {mat};
  gemv_flow_body<T, BITS, SIGNED, ZMODE, LATE, TILED, MX, TL, 1, NW>((int)blockIdx.x, x, mats, N, nullptr, 0, p);
}
// Several linears of the same m, k and quantisation: the grid is the concatenation of their blocks.
template<typename T, int BITS, bool SIGNED, int ZMODE, bool LATE, int MX, int TL, int NW>
__global__ void __launch_bounds__(NW * 64)
gemv_flow_grouped(GemvGroup g, FlowArgs p) {
  const GemvProblem pr = select_problem(g, (int)blockIdx.x);
  const RowsMat mats[1] = {{pr.w, static_cast<const uint16_t*>(pr.scale), static_cast<const uint16_t*>(pr.zero),
                            static_cast<const uint16_t*>(pr.bias), static_cast<uint16_t*>(pr.out)}};
  gemv_flow_body<T, BITS, SIGNED, ZMODE, LATE, false, MX, TL, 1, NW>((int)blockIdx.x - pr.first_block,
                                                              static_cast<const uint16_t*>(pr.x), mats, pr.N, nullptr,
                                                              0, p);
}
// hidden = x w^T + b -> out, gate = x v^T + c -> out2, y = hidden * act(gate): a block owns the same rows
// of both weights.
template<typename T, int BITS, bool SIGNED, int ZMODE, bool LATE, int MX, int TL, int NW>
__global__ void __launch_bounds__(NW * 64)
gemv_flow_glu(const uint16_t* __restrict__ x, RowsMat hidden, RowsMat gate, int N, uint16_t* __restrict__ y, int act,
              FlowArgs p) {
  const RowsMat mats[2] = {hidden, gate};
  gemv_flow_body<T, BITS, SIGNED, ZMODE, LATE, false, MX, TL, 2, NW>((int)blockIdx.x, x, mats, N, y, act, p);
}

}  // namespace
}  // namespace ofq
