// MFMA GEMM of fused_linear_with_groupwise_quantized_weight for a middling number of rows of x
// (17 to about 1000): the weights stay packed until they are in the registers of the wave that
// multiplies them.
//
// gemm_core2 (gemm_kernels.h) expands a weight tile into LDS for all its waves and fetches the codes
// through registers; with few rows of x its time is not the matrix instructions' but the wait, once
// per k-tile of 64, for codes that come from HBM.  Here
//   - a wave owns 32 columns of the output (32 weight rows) and ALL rows of the block's x tile
//     (TM * 32), so a code is expanded once per TM matrix instructions, by the lane that feeds it to
//     them, and never written back to LDS;
//   - x and the packed codes both arrive by asynchronous global -> LDS copies, in a ring of NSTAGE
//     stages; the only waits on memory are counted by hand and leave the younger stages in flight;
//   - KH waves share the columns and take alternate 64-element pieces of K (one step covers KH * 64
//     elements), added up through LDS at the end: more waves per CU without more columns per block;
//   - blocks split K further where the tiles do not fill the chip, writing fp32 partial sums as they
//     lie in the registers (1 KB per instruction); gemm_wr_fold adds them in order.
//
// Operand order.  A lane (n = lane % 32, half = lane / 32) reads the 16 bytes of codes (32 4-bit
// elements; 2 x 16 bytes of 8-bit ones) that belong to k = 32 * half .. 32 * half + 31 of the step's
// 64-element piece, and matrix instruction j of the piece takes its elements 8 j .. 8 j + 7: the sum
// over k does not mind the order as long as x follows it, i.e. x's 16-byte piece 4 * half + j of
// the 128-byte row.
//
// w~ = T(T(q) * s) + z with the reference's roundings (dequant_regs.h), products and sums in fp32 in
// the matrix core, one rounding of the result.
//
// What bounds it: for tall tiles the matrix cores with the conversions in their shadow and, once every CU
// has a block, what the blocks share: a step of 192 x 256 x 64 on symmetric fp16 4-bit codes takes 0.72 us
// in a block that is alone and 1.06 us in each of 256 (6.3 MFLOP a step: 1.5 PFLOP/s over the chip).  For
// flat tiles the fixed 6 us of two launches and the pipeline's start, the scales (1.9 us per 4096 of them,
// before the first step) and the partial sums.  The steps of every tile: wr_plan_us in gemm.hip.  Before
// and after (gemm_core2 above 64 rows, gemv_rows_mt below), us, fp16 4-bit:
//   64 x 4096 x 11008   28.2 -> 17.2     333 x 4096 x 11008          59.6 -> 47.7
//   64 x 32000 x 4096   46.2 -> 28.1     640 x 8192 x 8192 (zero)   143.7 -> 107.9
//   128 x 11008 x 4096  29.5 -> 23.7     900 x 11008 x 4096 (zero)  103.7 -> 88.4
#pragma once

#include "gemm_kernels.h"
#include "scale_panel.h"

namespace ofq {
namespace {

struct WrParams {
  const uint8_t* x;       // [M, K] T
  const uint8_t* w;       // [N, K * BITS / 8]
  const uint16_t* scale;  // [N, G]
  const uint16_t* zero;
  const uint16_t* bias;   // [N] or nullptr
  uint16_t* out;          // [M, N]
  float* part;            // K slices only: [splits][m32][n32][4][64][4]
  int M, N, K, G;
  uint32_t group_magic;               // ceil(2^32 / group_size): k / group_size is a multiply-high
  int group_size;
  int m_tiles, n_tiles;
  int steps_total, steps_per_split;   // steps of KH * 64 elements
  int panel_steps, panel_groups;      // scales in LDS at a time
};

template<int BITS>
constexpr int wr_code_bytes() { return 64 * BITS / 8; }  // of a row and a 64-element piece

template<int BITS, int TM, int WN, int KH>
constexpr size_t wr_stage_bytes() {
  return (size_t)TM * 32 * kStageRow * KH + (size_t)WN * 32 * wr_code_bytes<BITS>() * KH;
}

// 32 x 32 results of a wave (D[n][m]: lane = m % 32, quad g = n 8 g + 4 half .. + 3) -> T, through
// 32 rows of kPitch bytes of LDS, to rows of out
template<typename T>
__device__ __forceinline__ void wr_store_tile(const f32x16& acc, uint8_t* lds, uint16_t* out,
                                              const uint16_t* bias, int m0, int n0, int M, int N,
                                              int lane) {
  typedef typename TT<T>::storage S;
  constexpr int kPitch = 72;
  const int half = lane >> 5;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    S q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = n0 + 8 * g + 4 * half + e;
      float v = acc[4 * g + e];
      if (bias != nullptr) v += TT<T>::load(reinterpret_cast<const S*>(bias) + (n < N ? n : N - 1));
      TT<T>::store(&q[e], v);
    }
    *reinterpret_cast<u32x2*>(lds + (lane & 31) * kPitch + (8 * g + 4 * half) * 2) =
        *reinterpret_cast<const u32x2*>(q);
  }
  // (a wave reads what it wrote itself; its LDS operations complete in order)
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = i * 16 + (lane >> 2), piece = lane & 3;
    const u32x2 lo = *reinterpret_cast<const u32x2*>(lds + row * kPitch + piece * 16);
    const u32x2 hi = *reinterpret_cast<const u32x2*>(lds + row * kPitch + piece * 16 + 8);
    const u32x4 v = {lo[0], lo[1], hi[0], hi[1]};
    const int m = m0 + row, n = n0 + piece * 8;
    if (m < M) {
      uint16_t* dst = out + (int64_t)m * N + n;
      if (n + 8 <= N) {
        *reinterpret_cast<u32x4_any*>(dst) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (n + e < N) dst[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
        }
      }
    }
  }
}

// a pointer every lane agrees on, for the scalar operand of an asynchronous copy (the compiler
// loses track of it inside the per-lane branch of a ragged K)
__device__ __forceinline__ const uint8_t* wr_uniform(const uint8_t* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return reinterpret_cast<const uint8_t*>(((uint64_t)hi << 32) | lo);
}

template<int N>
__device__ __forceinline__ void wr_wait_and_barrier() {
  // this wave's copies but the N youngest have landed and its LDS reads are done, then everyone's
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template<typename T, class MF, int BITS, bool SIGNED, int ZMODE, int TM, int WN, int KH, int NSTAGE,
         bool RAGGED, bool SPLIT>
__global__ void __launch_bounds__(WN * KH * 64)
gemm_wr(WrParams p) {
  typedef typename TT<T>::storage S;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int W = WN * KH, NT = W * 64;
  constexpr int BM = TM * 32, BN = WN * 32;
  constexpr int kCB = wr_code_bytes<BITS>();
  constexpr int kCodeOps = kCB / 32;                 // copies of a wave's codes per step
  constexpr int kXBytes = BM * kStageRow * KH;
  constexpr int kStage = (int)wr_stage_bytes<BITS, TM, WN, KH>();
  // copies of x per step: KH * TM * 4 of 1 KB over W waves
  static_assert(kXBytes % (W * 1024) == 0, "every wave issues as many copies: its waits are one constant");
  constexpr int kXOps = kXBytes / (W * 1024);
  constexpr int kOps = kXOps + kCodeOps;
  // vector instructions between two matrix instructions: a quarter step's conversion over TM slots
  constexpr int kDequant = TT<T>::dtype == OFQ_BF16 ? (ZMODE == 0 ? 26 : 46) : (ZMODE == 0 ? 22 : 26);
  constexpr int kValu = (kDequant + TM - 1) / TM + 1;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, kh = wave / WN;

  // blocks of an XCD (block id mod 8) take neighbouring tiles, those of one K slice after another
  const int nblocks = gridDim.x;
  int logical;
  {
    const int b = blockIdx.x;
    const int xcd = b & 7, idx = b >> 3;
    const int per = nblocks >> 3, rem = nblocks & 7;
    logical = xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
  }
  const int tiles = p.m_tiles * p.n_tiles;
  const int split = SPLIT ? logical / tiles : 0;
  const int tile = SPLIT ? logical - split * tiles : logical;
  const int m0 = (tile % p.m_tiles) * BM;
  const int n0 = (tile / p.m_tiles) * BN;
  const int step0 = SPLIT ? split * p.steps_per_split : 0;
  int nsteps = p.steps_total - step0;
  if (SPLIT && nsteps > p.steps_per_split) nsteps = p.steps_per_split;

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const int K2 = p.K * 2;  // bytes of a row of x
  const int row_bytes = p.K * BITS / 8;

  // ---- copies: lane offsets that do not change from step to step ------------------------------
  // x: op o of this wave is 8-row group q = o * W + wave of the stage's KH * BM rows; lane (row
  // lane / 8, position lane % 8) fetches piece position ^ key of its row
  uint32_t xoff[kXOps];
  int xk[kXOps];  // byte of the row within the step
#pragma unroll
  for (int o = 0; o < kXOps; ++o) {
    const int q = o * W + wave;
    const int sub = q / (BM / 8);                 // which 64-element piece of the step
    const int rel = (q % (BM / 8)) * 8 + (lane >> 3);
    int row = m0 + rel;
    row = row < p.M ? row : p.M - 1;
    xk[o] = sub * kStageRow + (((lane & 7) ^ swizzle_key(rel)) << 4);
    xoff[o] = (uint32_t)(row - m0) * (uint32_t)K2 + (uint32_t)xk[o];
  }
  const uint8_t* xbase = p.x + (int64_t)m0 * K2;
  uint32_t woff[kCodeOps];
  int wk[kCodeOps];
#pragma unroll
  for (int o = 0; o < kCodeOps; ++o) {
    int row = n0 + wn * 32 + (lane & 31);
    row = row < p.N ? row : p.N - 1;
    wk[o] = kh * kCB + (lane >> 5) * (kCB / 2) + o * 16;
    woff[o] = (uint32_t)(row - n0) * (uint32_t)row_bytes + (uint32_t)wk[o];
  }
  const uint8_t* wbase = p.w + (int64_t)n0 * row_bytes;
  // copy o of step t into stage buf.  Steps past the block's last one repeat it (into a stage nobody
  // reads): every step then issues the same copies, its waits are one constant and its body has no
  // branch.
  auto issue_op = [&](int o, int t, int buf) {
    const int gs = step0 + (t < nsteps ? t : nsteps - 1);
    const uint32_t st = lds0 + (uint32_t)buf * kStage;
    if (o < kXOps) {
      const int q = o * W + wave;
      const uint8_t* src = wr_uniform(xbase + (int64_t)gs * (kStageRow * KH));
      if (!RAGGED || gs * (kStageRow * KH) + xk[o] < K2) {
        async_copy16_unordered(src, xoff[o], st + q * 1024);
      } else {
        *reinterpret_cast<u32x4*>(smem + buf * kStage + q * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
      }
    } else {
      const int c = o - kXOps;
      const uint8_t* src = wr_uniform(wbase + (int64_t)gs * (kCB * KH));
      uint32_t off = woff[c];
      // past the end of a ragged row: its first bytes of this step's piece 0 (their scale is zero)
      if (RAGGED && gs * (kCB * KH) + wk[c] >= row_bytes) off -= (uint32_t)wk[c];
      async_copy16_unordered(src, off, st + kXBytes + (wave * kCodeOps + c) * 1024);
    }
  };
  auto issue = [&](int t, int buf) {
#pragma unroll
    for (int o = 0; o < kOps; ++o) issue_op(o, t, buf);
  };
#pragma unroll
  for (int t = 0; t < NSTAGE - 1; ++t) issue(t, t);

  // ---- scales of the block's columns in LDS, [group][column], and a row of zeros behind them: the scale
  //      past the end of K, where x is zero but a code might overflow T under a group's scale, and
  //      infinity times zero is NaN ------------------------------------------------------------------
  uint16_t* sl = reinterpret_cast<uint16_t*>(smem + NSTAGE * kStage);
  uint16_t* zl = sl + (p.panel_groups + 1) * BN;
  int g0 = 0, ng = 0;  // groups in the panel
  auto group_of = [&](int k) { return (int)__umulhi((uint32_t)k, p.group_magic); };
  auto fill_panel = [&](int t) {
    g0 = group_of((step0 + t) * (KH * 64));
    ng = p.G - g0;
    ng = ng < p.panel_groups ? ng : p.panel_groups;
    copy_scale_panel<NT, ZMODE == 2, true>(p.scale + (int64_t)n0 * p.G + g0,
                                           p.zero + (int64_t)n0 * p.G + g0, p.G, BN, p.N - n0, ng,
                                           BN, sl, zl, tid);
    if (RAGGED && tid < BN) {
      sl[p.panel_groups * BN + tid] = 0;
      if (ZMODE == 2) zl[p.panel_groups * BN + tid] = 0;
    }
    __syncthreads();
  };

  f32x16 acc[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;

  const int half = lane >> 5;
  const int frag_row = lane & 31;
  const int x7 = swizzle_key(frag_row);
  const int xfrag = (kh * BM + frag_row) * kStageRow;
  const int col = wn * 32 + frag_row;

  // Software pipeline over the quarters j of a step: while the matrix instructions of a quarter
  // run, the wave reads the x operands of the next one and expands its codes; the codes and scales
  // of the next step are read in the second quarter.  So the first matrix instruction behind a
  // barrier has its operands in registers, and the barrier (which only says that stage t + 1 is
  // complete and the stage of t - 1 free) does not open a bubble of LDS latency and conversion.
  u32x4 a[2][TM], b[2];
  u32x4 codes[kCodeOps], codes_next[kCodeOps];
  float s, z, s_next, z_next;
  auto read_codes = [&](int t, int buf, u32x4 (&dst)[kCodeOps], float& sd, float& zd) {
    const uint8_t* cp = smem + buf * kStage + kXBytes + wave * (kCodeOps * 1024) + lane * 16;
#pragma unroll
    for (int o = 0; o < kCodeOps; ++o) dst[o] = *reinterpret_cast<const u32x4*>(cp + o * 1024);
    int g = group_of((step0 + t) * (KH * 64) + kh * 64 + half * 32) - g0;
    g = g < ng ? g : (RAGGED ? p.panel_groups : 0);  // (past the panel: not used)
    sd = TT<T>::load(reinterpret_cast<const S*>(sl) + g * BN + col);
    zd = 0.f;
    if (ZMODE == 2) zd = TT<T>::load(reinterpret_cast<const S*>(zl) + g * BN + col);
    if (ZMODE == 1) zd = TT<T>::round(-(float)((1 << (BITS - 1)) - 1) * sd);
  };
  auto read_x = [&](int buf, int j, u32x4 (&dst)[TM]) {
    const uint8_t* st = smem + buf * kStage + xfrag + (((4 * half + j) ^ x7) << 4);
#pragma unroll
    for (int i = 0; i < TM; ++i) dst[i] = *reinterpret_cast<const u32x4*>(st + i * (32 * kStageRow));
  };
  auto expand = [&](const u32x4 (&c)[kCodeOps], int j, float sv, float zv) {
    if constexpr (BITS == 4) {
      return dequant8_b4<T, SIGNED, ZMODE>(c[0][j], sv, zv);
    } else {
      return dequant8_b8<T, SIGNED, ZMODE>(c[j >> 1][2 * (j & 1)], c[j >> 1][2 * (j & 1) + 1], sv, zv);
    }
  };
  int buf = 0;
  auto step = [&](int t) {
    // stages up to t + 1 are complete: all but the copies of the NSTAGE - 3 younger ones (none may be
    // left in flight where a ragged K's last stage has fewer copies)
    if (RAGGED) {
      wr_wait_and_barrier<0>();
    } else {
      wr_wait_and_barrier<kOps * (NSTAGE - 3)>();
    }
    const int free_buf = buf == 0 ? NSTAGE - 1 : buf - 1;
    const int next_buf = buf + 1 == NSTAGE ? 0 : buf + 1;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int cur = j & 1, nxt = cur ^ 1;
      if (j < 3) {
        read_x(buf, j + 1, a[nxt]);
      } else {
        read_x(next_buf, 0, a[nxt]);
      }
      if (j == 1) read_codes(t + 1, next_buf, codes_next, s_next, z_next);
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[i] = MF::mma(b[cur], a[cur][i], acc[i]);
#pragma unroll
      for (int o = j * kOps / 4; o < (j + 1) * kOps / 4; ++o) issue_op(o, t + NSTAGE - 1, free_buf);
      b[nxt] = j < 3 ? expand(codes, j + 1, s, z) : expand(codes_next, 0, s_next, z_next);
      // Interleaved by hand: a matrix instruction occupies its pipe for 32 clocks and the wave issues
      // in order, so the conversions have to stand between the matrix instructions to run in their
      // shadow; behind them, the waves of a block, which the barrier keeps in step, all convert at
      // the same time with the matrix pipes idle.
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // matrix
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
        __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
      }
    }
#pragma unroll
    for (int o = 0; o < kCodeOps; ++o) codes[o] = codes_next[o];
    s = s_next;
    z = z_next;
    buf = next_buf;
  };
  for (int first = 0; first < nsteps; first += p.panel_steps) {
    if (first > 0) __syncthreads();  // everyone is done with the panel before
    fill_panel(first);
    if (first == 0) wr_wait_and_barrier<0>();  // stage 0
    read_codes(first, buf, codes, s, z);
    read_x(buf, 0, a[0]);
    b[0] = expand(codes, 0, s, z);
    const int last = nsteps - first < p.panel_steps ? nsteps : first + p.panel_steps;
    for (int t = first; t < last; ++t) step(t);
  }

  // ---- add up the K pieces of the block, then store --------------------------------------------
  wr_wait_and_barrier<0>();  // the copies issued past the end have landed, the stages are free
  if constexpr (KH > 1) {
    f32x4* red = reinterpret_cast<f32x4*>(smem);  // [KH - 1][WN][TM][4][64]
    constexpr int kAll = (int)(NSTAGE * wr_stage_bytes<BITS, TM, WN, KH>());
    static_assert((KH - 1) * WN * TM * 4096 <= kAll, "the sums of the K pieces fit the stages");
    if (kh > 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          red[((((kh - 1) * WN + wn) * TM + i) * 4 + g) * 64 + lane] =
              f32x4{acc[i][4 * g], acc[i][4 * g + 1], acc[i][4 * g + 2], acc[i][4 * g + 3]};
        }
    }
    __syncthreads();
    if (kh == 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int h = 0; h < KH - 1; ++h)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 v = red[(((h * WN + wn) * TM + i) * 4 + g) * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][4 * g + e] += v[e];
          }
    }
    if (!SPLIT) __syncthreads();  // the sums are read; the output goes through the same memory
    if (kh > 0) return;
  }
  const int nw0 = n0 + wn * 32;
  if (nw0 >= p.N) return;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int mi = m0 + i * 32;
    if (mi >= p.M) break;
    if constexpr (SPLIT) {
      const int m32 = (p.M + 31) >> 5, n32 = (p.N + 31) >> 5;
      float* dst = p.part + ((((int64_t)split * m32 + (mi >> 5)) * n32 + (nw0 >> 5)) * 4) * 256 + lane * 4;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        *reinterpret_cast<f32x4*>(dst + g * 256) =
            f32x4{acc[i][4 * g], acc[i][4 * g + 1], acc[i][4 * g + 2], acc[i][4 * g + 3]};
      }
    } else {
      wr_store_tile<T>(acc[i], smem + wn * 2304, p.out, p.bias, mi, nw0, p.M, p.N, lane);
    }
  }
}

// Adds the K slices of a 32 x 32 tile in order, adds the bias and rounds once.  A block is a tile, a
// wave one quad of its rows of weights; the slices are requested together.
template<typename T>
__global__ void __launch_bounds__(256)
gemm_wr_fold(const float* __restrict__ part, const uint16_t* __restrict__ bias,
             uint16_t* __restrict__ out, int M, int N, int splits) {
  typedef typename TT<T>::storage S;
  constexpr int kPitch = 72;
  constexpr int U = 8;
  __shared__ __attribute__((aligned(16))) uint8_t lds[32 * kPitch];
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int m32 = (M + 31) >> 5, n32 = (N + 31) >> 5;
  const int tile = blockIdx.x;
  const int64_t slice = (int64_t)m32 * n32 * 1024;
  const float* src = part + (int64_t)tile * 1024 + g * 256 + lane * 4;
  const int m0 = (tile / n32) * 32, n0 = (tile % n32) * 32;
  const int nl = 8 * g + 4 * (lane >> 5);
  S bv[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int n = n0 + nl + e;
    if (bias != nullptr) bv[e] = reinterpret_cast<const S*>(bias)[n < N ? n : N - 1];
  }
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < splits; s0 += U) {
    f32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u < splits ? s0 + u : splits - 1;
      v[u] = *reinterpret_cast<const f32x4*>(src + s * slice);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s0 + u < splits) sum = s0 + u == 0 ? v[u] : sum + v[u];
    }
  }
  S q[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float v = sum[e];
    if (bias != nullptr) v += TT<T>::load(&bv[e]);
    TT<T>::store(&q[e], v);
  }
  *reinterpret_cast<u32x2*>(lds + (lane & 31) * kPitch + nl * 2) = *reinterpret_cast<const u32x2*>(q);
  __syncthreads();
  // 32 rows x 64 bytes: 8 bytes a thread
  const int row = threadIdx.x >> 3, piece = threadIdx.x & 7;
  const u32x2 v = *reinterpret_cast<const u32x2*>(lds + row * kPitch + piece * 8);
  const int m = m0 + row, n = n0 + piece * 4;
  if (m < M) {
    uint16_t* dst = out + (int64_t)m * N + n;
    if (n + 4 <= N) {
      *reinterpret_cast<u32x2_any*>(dst) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (n + e < N) dst[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
      }
    }
  }
}

}  // namespace
}  // namespace ofq
