// Streaming kernel of fused_linear_with_groupwise_quantized_weight for 17 to 64 rows of x, fp16 and bf16, 4-
// and 8-bit codes, groups along K: one linear, several in one launch, or the two of a gated linear unit with
// its gating.  Roundings, formats and ragged rows of K as in gemv_ring.h.
//
// Every CU needs all of x for its rows of the weight: 100 MB out of L2 for 48 x 11008 x 4096, four times what
// the codes bring.  Four of a block's 16 waves, one on every SIMD, do nothing but copy x, up to three buffers of LDS
// ahead; they wait for it, the others do not.  Twelve waves expand and multiply: groups over the tiles
// of 16 rows, sharing K within a group, 1, 2, 3, 4, 6 or 12 waves as the host picks.  Their codes come by
// counted asynchronous copies, up to three steps ahead: a wave's copies complete in order, so that codes from
// HBM behind copies of x, or in front of them, would be waited for at every barrier -- hence the split.
//
// What bounds it: a phase (one step of every wave between two barriers), the way from the barrier over x from LDS,
// the expansion and the products to the next one, and 5.5 us to start, load the first x, fold and store.  A phase takes
// 1.3 to 1.5 us where a wave has one tile of 4-bit codes (n = 11008, weights from HBM: 8.2, 11.0 and 16.8 us for 2, 4
// and 8 phases at 48 rows, 8.6, 11.5 and 18.4 at 64).  Its x is read from LDS by every wave for its own tiles, so more
// tiles of a wave cost less each.  Waves wait for 60 % of their lives at 48 x 11008 x 4096, LDS is busy 38 % of the
// time, more than half of that with conflicts of banks, vector units 47 %, matrix units 13 %, L2 serves 7 TB/s.
// Against gemv_rows_mt (us):
//   fp16 4-bit  48 x 11008 x 4096 with a zero point  17.8 -> 16.0   64 x 11008 x 4096        20.6 -> 18.6
//   fp16 4-bit  40 x 22000 x 2944   29.3 -> 18.2 (gemm_wr 19.9)     20 x 2 x 9216 x 3584     27.3 -> 18.7
//   8 bits      56 x 2 x 12032 x 3968 bf16  51.4 -> 33.2            45 x 2 x 10880 x 4096 fp16  43.2 -> 26
// Addresses of x made once instead of for every copy, and two to three buffers in flight: 48 x 11008 x 4096 21.2 -> 16.7.
// Codes and scales read from LDS a step ahead, in front of the barrier: 16.9 (not kept).
#pragma once

#include "gemv_ring.h"

namespace ofq {
namespace {

constexpr int kRingMtWorkers = 12;
constexpr int kRingMtCopiers = kRingWaves - kRingMtWorkers;
constexpr int kRingMtCopies = 16;   // of a copier for a buffer of x, at most

// all but the n youngest copies have landed (or a few more)
__device__ __forceinline__ void ring_mt_wait(int n) {
  switch (n >> 2) {
    case 0: wait_vmem_all(); break;
    case 1: wait_vmem_le<4>(); break;
    case 2: wait_vmem_le<8>(); break;
    case 3: wait_vmem_le<12>(); break;
    case 4: wait_vmem_le<16>(); break;
    case 5: wait_vmem_le<20>(); break;
    case 6: wait_vmem_le<24>(); break;
    case 7: wait_vmem_le<28>(); break;
    default: wait_vmem_le<32>(); break;
  }
}

struct RingMtArgs {
  int M, K, group_size, gs_shift;
  int rows_per_block;
  int wk;           // workers = (12 / wk) groups over the tiles x wk over K
  int depth;        // steps of codes ahead, depth * tiles of a wave <= 4
  int buffers;      // of x in LDS, of wk steps each
  int phases;       // ceil(steps / wk)
  uint32_t m_magic;  // ceil(2^32 / M)
};

// the partial sums of one output, in order
template<int WK>
__device__ __forceinline__ float ring_mt_sum(const float* src, int stride) {
  float part[WK];
#pragma unroll
  for (int q = 0; q < WK; ++q) part[q] = src[q * stride];
  float v = 0.f;
#pragma unroll
  for (int q = 0; q < WK; ++q) v += part[q];
  return v;
}

template<typename T, int BITS, bool SIGNED, int ZMODE, int MT, int TL, int NMAT>
__device__ __forceinline__ void
gemv_ring_mt_body(int block, const uint16_t* __restrict__ x, const RowsMat (&mats)[NMAT], int N,
                  uint16_t* __restrict__ y, int act, const RingMtArgs& p) {
  typedef typename TT<T>::storage S;
  static_assert(sizeof(S) == 2, "16-bit element types");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int CK = BITS == 4 ? 128 : 64;  // elements per chunk: 64 bytes of codes per row
  constexpr int LK = CK / 4;                // elements per lane and chunk
  constexpr int XV = LK / 8;                // 16-byte pieces of x per lane and chunk
  constexpr int kRec = CK * 2;              // bytes of x of one row and chunk
  constexpr int kPieces = kRec / 16;
  constexpr int kMaxDepth = TL == 1 ? 3 : (TL == 2 ? 2 : 1);
  constexpr int kRegions = ZMODE == kZeroAsym ? 2 : 1;
  const int M = p.M, K = p.K;
  const int row_bytes = K / LK * 16;
  const int G = p.gs_shift >= 0 ? K >> p.gs_shift : K / p.group_size;
  const int steps = (K + CK - 1) / CK;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int WK = p.wk;
  const int wt = wave / WK, wk = wave - wt * WK;
  const int r = lane & 15;
  const int kb = lane >> 4;
  const int row0 = block * p.rows_per_block;
  int rows_blk = N - row0;
  if (rows_blk > p.rows_per_block) rows_blk = p.rows_per_block;
  if (rows_blk <= 0) return;
  const int ntiles = (rows_blk + 15) >> 4;  // per matrix
  const int nvt = NMAT * ntiles;

  // LDS: [scales, zeros of every matrix][rings of the workers][two to four buffers of x]; the sums take the
  //      place of all of it
  const int sreg = ring_scale_bytes(p.rows_per_block, G);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const int rings = (NMAT * kRegions * sreg + 1023) & ~1023;
  const int xbase = rings + kRingMtWorkers * (p.depth * TL * 1024);
  const int xbuf_bytes = (WK * M * kRec + 1023) & ~1023;

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

  f32x4 acc[TL][MT];
#pragma unroll
  for (int t = 0; t < TL; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // pieces of a record are swizzled so that the 16 rows of an operand read meet different banks
  auto swizzle = [](int m) { return BITS == 4 ? m & 15 : (m >> 1) & 7; };
  // (every barrier below is passed by both kinds of waves, 1 + (phases - 1) times)
  if (wave >= kRingMtWorkers) {
    const int copier = wave - kRingMtWorkers;
#pragma unroll
    for (int i = 0; i < NMAT * kRegions; ++i) {
      const RowsMat& mt = mats[i / kRegions];
      const uint8_t* src = reinterpret_cast<const uint8_t*>(i % kRegions == 0 ? mt.scale : mt.zero)
                           + (s_first - s_shift);
      const int nops = (s_bytes + 1023) >> 10;
      for (int op = copier; op < nops; op += kRingMtCopiers) {
        const int o = op * 1024 + lane * 16;
        if (o < s_bytes && s_first - s_shift + o + 16 <= all_bytes) {
          async_copy16_at(src, (uint32_t)o, lds0 + i * sreg + op * 1024);
        }
      }
    }
    // a phase: records of 1 row and chunk, chunk by chunk
    const int full_ops = (WK * M * kRec + 1023) >> 10;
    uint32_t off[kRingMtCopies];  // of this lane, in a phase that K fills
#pragma unroll
    for (int i = 0; i < kRingMtCopies; ++i) {
      const int rec = (copier + i * kRingMtCopiers) * (1024 / kRec) + lane / kPieces;
      const int c = (int)__umulhi((uint32_t)rec, p.m_magic);
      const int m = rec - c * M;
      const uint32_t at = (uint32_t)m * (uint32_t)(K * 2) + (uint32_t)(c * kRec + (((lane % kPieces) ^ swizzle(m)) << 4));
      off[i] = rec < WK * M ? at : 0u;  // (beyond: the rest of the buffer's last KB)
    }
    auto phase_ops = [&](int phase) {  // of this wave
      const int left = steps - phase * WK;
      const int ops = left < WK ? (left * M * kRec + 1023) >> 10 : full_ops;
      return ops <= copier ? 0 : (ops - copier + kRingMtCopiers - 1) / kRingMtCopiers;
    };
    auto copy_x = [&](int phase, int buffer) {
      const uint32_t to = lds0 + xbase + buffer * xbuf_bytes;
      const int c0 = phase * WK;
      if ((c0 + WK) * CK <= K) {
        const uint8_t* src = reinterpret_cast<const uint8_t*>(x) + (size_t)c0 * kRec;
#pragma unroll
        for (int i = 0; i < kRingMtCopies; ++i) {
          const int op = copier + i * kRingMtCopiers;
          if (op < full_ops) async_copy16_at(src, off[i], to + op * 1024);
        }
        return;
      }
      const int left = steps - c0;
      const int nrec = (left < WK ? left : WK) * M;
      for (int op = copier; op < (nrec * kRec + 1023) >> 10; op += kRingMtCopiers) {
        const int rec = op * (1024 / kRec) + lane / kPieces;
        const int c = (int)__umulhi((uint32_t)rec, p.m_magic);
        const int m = rec - c * M;
        const int byte = (c0 + c) * kRec + (((lane % kPieces) ^ swizzle(m)) << 4);
        // (some lane of every copy has bytes to bring: the first record's first piece)
        if (rec < nrec && byte < K * 2) {
          async_copy16_at(reinterpret_cast<const uint8_t*>(x), (uint32_t)m * (uint32_t)(K * 2) + (uint32_t)byte,
                          to + op * 1024);
        } else {
          *reinterpret_cast<u32x4*>(smem + (to - lds0) + op * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
        }
      }
    };
    for (int phase = 0; phase + 1 < p.buffers && phase < p.phases; ++phase) copy_x(phase, phase);
    int into = p.buffers - 1;
    for (int phase = 0; phase < p.phases; ++phase) {
      int younger = 0;
      for (int q = phase + 1; q < phase + p.buffers - 1 && q < p.phases; ++q) younger += phase_ops(q);
      ring_mt_wait(younger);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      // (the readers of the buffer that comes next have passed that barrier)
      if (phase + p.buffers - 1 < p.phases) copy_x(phase + p.buffers - 1, into);
      into = into + 1 == p.buffers ? 0 : into + 1;
    }
  } else {
    const int end = wt * TL < nvt ? steps : 0;  // a group beyond the tiles has nothing to do
    uint32_t roff[TL];         // of this lane's row of every tile, and its place in a chunk
    const uint8_t* wbase[TL];  // (the same for every lane)
    int srow[TL];              // LDS bytes of its scales
#pragma unroll
    for (int t = 0; t < TL; ++t) {
      const int vt = wt * TL + t;
      const bool second = NMAT == 2 && vt >= ntiles;
      const int row_l = (second ? vt - ntiles : vt) * 16 + r;
      const bool ok = vt < nvt && row_l < rows_blk;
      roff[t] = (ok ? (uint32_t)row_l * (uint32_t)row_bytes : 0u) + (uint32_t)(kb * 16);
      wbase[t] = mats[NMAT == 2 && second ? NMAT - 1 : 0].w + (int64_t)row0 * row_bytes;
      srow[t] = (second ? kRegions * sreg : 0) + s_shift + (ok ? row_l : 0) * G * 2;
    }
    const int ring0 = rings + wave * (p.depth * TL * 1024);
    // codes of a step's tile; bytes past the row's end re-read the step's first ones
    auto copy_codes = [&](int s, int slot, int t) {
      const uint32_t at = (uint32_t)s * 64u;
      uint32_t off = roff[t];
      if ((int)at + 64 > row_bytes) {  // (the same for every lane)
        if ((int)at + kb * 16 >= row_bytes) off -= (uint32_t)(kb * 16);
      }
      async_copy16_at(wbase[t] + at, off, lds0 + ring0 + (slot * TL + t) * 1024);
    };
    // of this wave's steps from s on, how many are among the next n
    auto live_steps = [&](int s, int n) {
      int live = 0;
#pragma unroll
      for (int d = 0; d < kMaxDepth; ++d) live += d < n && s + d * WK < end ? 1 : 0;
      return live;
    };
#pragma unroll
    for (int d = 0; d < kMaxDepth; ++d) {
      if (d < p.depth && wk + d * WK < end) {
#pragma unroll
        for (int t = 0; t < TL; ++t) copy_codes(wk + d * WK, d, t);
      }
    }
    // this lane's pieces of x within a chunk: row r of each tile of x (rows >= M of the last one repeat row
    // M - 1 and feed results that are nobody's)
    int xoff[XV], xlast[XV];
    {
      const int ml = (MT - 1) * 16 + r < M ? (MT - 1) * 16 + r : M - 1;
#pragma unroll
      for (int j = 0; j < XV; ++j) {
        xoff[j] = r * kRec + (((kb * XV + j) ^ swizzle(r)) << 4);
        xlast[j] = ml * kRec + (((kb * XV + j) ^ swizzle(ml)) << 4);
      }
    }
    int slot = 0, from = 0;
    u32x4 codes[TL];
    float sc[TL], z[TL];
    // codes, scales and zero points of step s into registers
    auto fetch = [&](int s) {
      int k0 = s * CK + kb * LK;
      const bool in_row = k0 < K;
      k0 = in_row ? k0 : 0;
      const int grp = p.gs_shift >= 0 ? (k0 >> p.gs_shift) : (k0 / p.group_size);
      const bool more = s + p.depth * WK < end;
      const int younger = live_steps(s + WK, p.depth - 1) * TL + TL - 1;
      const uint8_t* cp = smem + ring0 + slot * (TL * 1024) + lane * 16;
#pragma unroll
      for (int t = 0; t < TL; ++t) {
        // younger than this tile's copy: those of later steps, of the step's later tiles, and, if there
        // is such a step, what has taken the slots of its earlier tiles
        ring_wait(more ? younger : younger - t);
        asm volatile("" ::: "memory");
        codes[t] = *reinterpret_cast<const u32x4*>(cp + t * 1024);
        const uint16_t sraw = *reinterpret_cast<const uint16_t*>(smem + srow[t] + grp * 2);
        uint16_t zraw = 0;
        if (ZMODE == kZeroAsym) zraw = *reinterpret_cast<const uint16_t*>(smem + srow[t] + sreg + grp * 2);
        // the codes are in registers: their slot is free
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (more) copy_codes(s + p.depth * WK, slot, t);
        sc[t] = in_row ? raw16_to_float<T>(sraw) : 0.f;
        z[t] = 0.f;
        if (ZMODE == kZeroAsym) z[t] = in_row ? raw16_to_float<T>(zraw) : 0.f;
        if (ZMODE == kZeroSymU) z[t] = TT<T>::round(-(float)((1 << (BITS - 1)) - 1) * sc[t]);
      }
      slot = slot + 1 == p.depth ? 0 : slot + 1;
    };
    for (int s = wk, phase = 0; phase < p.phases; ++phase, s += WK) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (s < end) {
        fetch(s);
        const uint8_t* xp = smem + xbase + from * xbuf_bytes + wk * (M * kRec);
        auto x_piece = [&](int mt, int j) {
          return *reinterpret_cast<const u32x4*>(xp + (mt < MT - 1 ? mt * 16 * kRec + xoff[j] : xlast[j]));
        };
        if constexpr (BITS == 4) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            u32x4 xa[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) xa[mt] = x_piece(mt, j);
#pragma unroll
            for (int t = 0; t < TL; ++t) {
              if (wt * TL + t < nvt) {
                const u32x4 b = dequant8_b4<T, SIGNED, ZMODE>(codes[t][j], sc[t], z[t]);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[t][mt] = MfmaK32<T>::mma(xa[mt], b, acc[t][mt]);
              }
            }
          }
        } else {
          u32x4 xa[MT][2];
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            xa[mt][0] = x_piece(mt, 0);
            xa[mt][1] = x_piece(mt, 1);
          }
#pragma unroll
          for (int t = 0; t < TL; ++t) {
            if (wt * TL + t < nvt) {
              u32x4 b0, b1;
              dequant16_b8<T, SIGNED, ZMODE>(codes[t], sc[t], z[t], b0, b1);
#pragma unroll
              for (int mt = 0; mt < MT; ++mt) acc[t][mt] = MfmaK32<T>::mma(xa[mt][0], b0, acc[t][mt]);
#pragma unroll
              for (int mt = 0; mt < MT; ++mt) acc[t][mt] = MfmaK32<T>::mma(xa[mt][1], b1, acc[t][mt]);
            }
          }
        }
      }
      from = from + 1 == p.buffers ? 0 : from + 1;
    }
  }

  // ---- sums of the workers -> LDS, [tile][wave of K][M][16] -----------------------------------------
  __syncthreads();
  float* red = reinterpret_cast<float*>(smem);
  if (wave < kRingMtWorkers) {
#pragma unroll
    for (int t = 0; t < TL; ++t) {
      const int vt = wt * TL + t;
      if (vt < nvt) {
        float* dst = red + (size_t)(vt * WK + wk) * (M * 16);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int m = mt * 16 + 4 * kb + v;
            if (m < M) dst[m * 16 + r] = acc[t][mt][v];
          }
        }
      }
    }
  }
  __syncthreads();
  const int padded = ntiles * 16;
  for (int o = tid; o < M * padded; o += kRingWaves * 64) {
    const int m = o / padded;
    const int row_l = o - m * padded;
    if (row_l < rows_blk) {
      const int64_t at = (int64_t)m * N + row0 + row_l;
      S res[NMAT];
#pragma unroll
      for (int mt = 0; mt < NMAT; ++mt) {
        const float* src = red + (size_t)((mt * ntiles + (row_l >> 4)) * WK) * (M * 16) + m * 16 + (row_l & 15);
        float v;
        switch (WK) {  // (unrolled: the reads of a sum go out together)
          case 12: v = ring_mt_sum<12>(src, M * 16); break;
          case 6: v = ring_mt_sum<6>(src, M * 16); break;
          case 4: v = ring_mt_sum<4>(src, M * 16); break;
          case 3: v = ring_mt_sum<3>(src, M * 16); break;
          case 2: v = ring_mt_sum<2>(src, M * 16); break;
          default: v = ring_mt_sum<1>(src, M * 16); break;
        }
        if (mats[mt].bias != nullptr) {
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

template<typename T, int BITS, bool SIGNED, int ZMODE, int MT, int TL>
__global__ void __launch_bounds__(kRingWaves * 64)
gemv_ring_mt(const uint16_t* __restrict__ x, RowsMat mat, int N, RingMtArgs p) {
  const RowsMat mats[1] = {mat};
  gemv_ring_mt_body<T, BITS, SIGNED, ZMODE, MT, TL, 1>((int)blockIdx.x, x, mats, N, nullptr, 0, p);
}
// Several linears of the same m, k and quantisation: the grid is the concatenation of their blocks.
template<typename T, int BITS, bool SIGNED, int ZMODE, int MT, int TL>
__global__ void __launch_bounds__(kRingWaves * 64)
gemv_ring_mt_grouped(GemvGroup g, RingMtArgs p) {
  const GemvProblem pr = select_problem(g, (int)blockIdx.x);
  const RowsMat mats[1] = {{pr.w, static_cast<const uint16_t*>(pr.scale), static_cast<const uint16_t*>(pr.zero),
                            static_cast<const uint16_t*>(pr.bias), static_cast<uint16_t*>(pr.out)}};
  gemv_ring_mt_body<T, BITS, SIGNED, ZMODE, MT, TL, 1>((int)blockIdx.x - pr.first_block,
                                                       static_cast<const uint16_t*>(pr.x), mats, pr.N,
                                                       nullptr, 0, p);
}
// hidden = x w^T + b -> out, gate = x v^T + c -> out2, y = hidden * act(gate): a block owns the same rows
// of both weights.
template<typename T, int BITS, bool SIGNED, int ZMODE, int MT, int TL>
__global__ void __launch_bounds__(kRingWaves * 64)
gemv_ring_mt_glu(const uint16_t* __restrict__ x, RowsMat hidden, RowsMat gate, int N,
                 uint16_t* __restrict__ y, int act, RingMtArgs p) {
  const RowsMat mats[2] = {hidden, gate};
  gemv_ring_mt_body<T, BITS, SIGNED, ZMODE, MT, TL, 2>((int)blockIdx.x, x, mats, N, y, act, p);
}

}  // namespace
}  // namespace ofq
