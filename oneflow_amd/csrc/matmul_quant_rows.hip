// matmul_quant with few rows of a (m <= 96): int8 x int8 on v_mfma_i32_16x16x64_i8 with the weights
// streamed from HBM once.
//
// The tiled GEMM needs 128-row tiles to earn its LDS traffic and leaves most CUs without a block when a has a
// handful of rows; here a block owns consecutive rows of b (about n / 256, at most 64) and all of K.
//
// matmul_quant_stream.  The waves of a block share nothing until the end: a wave takes every eighth 128-byte step
// of K, and both its columns of a and its columns of the block's rows of b come by asynchronous global -> LDS
// copies into a ring of its own, D steps ahead, so there is no barrier in the loop and no request waits in a
// register.  A copy is 8 rows x 128 bytes: whole lines, where an operand request of the matrix instruction
// (16 rows x 64 bytes) takes half of each; the pieces of a row are XOR-swizzled on the way, so that the operand
// reads have no conflicts of banks.  Rows come in eights (a: MX, b: WX of them), rows past the end re-read the last
// one and feed results that are never stored.  int32 sums are added across the waves through LDS (integer addition: the
// order cannot matter) and leave through the epilogue of the GEMM path,
//   out = T(float(acc) * (a_scale * b_scale[n]) + bias[n]),
// so all paths give the same bits.
//
// What bounds it: up to 16 rows of a the stream of b (8 x 11008 x 4096: 9.7 us with weights from HBM, 45 MB at 6.2 TB/s
// behind 2.4 us of launch, first bytes and fold), beyond that b and the rows of a that every block reads from L2 together
// (64 x 11008 x 4096: 14.4 us; a CU takes in 50 to 60 bytes per ns).  Two, three or six steps ahead are the same
// within 3 %.  Codes waiting in registers, one request ahead and a from L2 in 64-byte runs, the kernel that this one
// took the place of: 12.8 and 21.9 us; 48 x 1024 x 2048 6.6 -> 4.5, 20 x 600 x 8192 11.5 -> 6.4, 24 x 4096 x 11008
// 18.9 -> 12.8.
#include <algorithm>
#include <atomic>
#include <cmath>
#include "gemm_kernels.h"
#include "ofq_device.h"
#include "ofq_internal.h"

namespace ofq {
namespace {

constexpr int kMqWaves = 8;      // 20 KB of LDS each
constexpr int kMqMaxM = 96;      // rows of a
// rows of b in a block (above 64 rows of a: what leaves room for the sums of the waves)
constexpr int mq_max_rows(int m) { return m > 64 ? 48 : 64; }

// steps of STEP KB that a wave holds or has requested
constexpr int mq_depth(int step_kb) { return 20 / step_kb > 3 ? 3 : 20 / step_kb; }

// all but the youngest n steps of STEP copies have landed
template<int STEP>
__device__ __forceinline__ void wait_steps(int n) {
  switch (n) {
    case 0: wait_vmem_all(); break;
    case 1: wait_vmem_le<STEP>(); break;
    default: wait_vmem_le<2 * STEP>(); break;
  }
}

struct MqStreamArgs {
  const float* a_scale;
  const float* b_scale;
  const void* bias;
  void* out;
  int out_dtype;
  int M, N, K;
  int rows_per_block;
};

template<typename T>
__device__ __forceinline__ void mq_store(const MqStreamArgs& p, int64_t at, float v, bool has_bias, float bias) {
  if (has_bias) v = v + bias;
  TT<T>::store(static_cast<typename TT<T>::storage*>(p.out) + at, v);
}

template<int MX, int WX>
__global__ void __launch_bounds__(kMqWaves * 64)
matmul_quant_stream(const uint8_t* __restrict__ a, const uint8_t* __restrict__ b, MqStreamArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int STEP = MX + WX, D = mq_depth(STEP);
  constexpr int MT = (MX + 1) / 2, WT = (WX + 1) / 2;  // 16-row tiles
  constexpr int R = WT * 16;
  static_assert(D >= 1 && D * STEP <= 20 && STEP * (D - 1) < 63, "LDS of a wave, vmcnt");
  const int M = p.M, N = p.N, K = p.K;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = blockIdx.x * p.rows_per_block;
  int rows_blk = N - row0;
  if (rows_blk > p.rows_per_block) rows_blk = p.rows_per_block;
  if (rows_blk <= 0) return;
  const int steps = (K + 127) >> 7;

  // a thread's outputs are those of one row of b: its scale and the bits of its bias are requested before the
  // copies, without a branch (the compiler waits at the end of one), and first looked at when the sums are there
  const int orow = tid % R;
  const int brow = row0 + (orow < rows_blk ? orow : 0);
  const float sa = p.a_scale[0];
  float sb = p.b_scale[brow];
  const bool has_bias = p.bias != nullptr, wide = p.out_dtype == OFQ_F32;
  const uint16_t* bias_at = static_cast<const uint16_t*>(has_bias ? p.bias : static_cast<const void*>(p.b_scale))
                            + (wide ? 2 * (int64_t)brow : brow);
  uint32_t bias_lo = bias_at[0], bias_hi = bias_at[wide ? 1 : 0];

  // ---- copies -----------------------------------------------------------------------------------
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem
                        + (uint32_t)wave * (D * STEP * 1024);
  const int sub = lane >> 3;                    // row of the eight
  const uint32_t piece = (uint32_t)(((lane & 7) ^ sub) << 4);
  uint32_t aoff[MX], boff[WX];                  // of this lane's row in every eight; rows past the end: the last one
#pragma unroll
  for (int i = 0; i < MX; ++i) aoff[i] = (uint32_t)(i * 8 + sub < M ? i * 8 + sub : M - 1) * (uint32_t)K + piece;
#pragma unroll
  for (int i = 0; i < WX; ++i) {
    boff[i] = (uint32_t)(i * 8 + sub < rows_blk ? i * 8 + sub : rows_blk - 1) * (uint32_t)K + piece;
  }
  const uint8_t* const bblk = b + (int64_t)row0 * K;
  auto copy_step = [&](int s, int slot) {
    const uint32_t lds = lds0 + (uint32_t)slot * (STEP * 1024);
    // the second half of the last step of a row of 64 (2 i + 1) bytes re-reads the first
    const uint32_t back = s * 128 + 64 >= K && piece >= 64 ? 64u : 0u;
    const uint8_t* as = a + s * 128;
    const uint8_t* bs = bblk + s * 128;
#pragma unroll
    for (int i = 0; i < MX; ++i) {
      async_copy16_at(as, aoff[i] - back, lds + i * 1024);
    }
#pragma unroll
    for (int i = 0; i < WX; ++i) {
      async_copy16_once(bs, boff[i] - back, lds + (MX + i) * 1024);
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (wave + d * kMqWaves < steps) copy_step(wave + d * kMqWaves, d);

  // ---- products ---------------------------------------------------------------------------------
  const int r = lane & 15, kb = lane >> 4;
  // this lane's piece of row r of a tile, in the two halves of a step; a tile of one eight has its rows twice
  const int at0 = (r & 7) * 128 + ((kb ^ (r & 7)) << 4), at1 = (r & 7) * 128 + (((4 + kb) ^ (r & 7)) << 4);
  const int upper = (r >> 3) * 1024;
  i32x4 acc[WT][MT];
#pragma unroll
  for (int t = 0; t < WT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = i32x4{0, 0, 0, 0};

  int slot = 0;
  for (int s = wave; s < steps; s += kMqWaves) {
    int live = 0;  // later steps under way
#pragma unroll
    for (int d = 1; d < D; ++d) live += s + d * kMqWaves < steps ? 1 : 0;
    wait_steps<STEP>(live);
    asm volatile("" ::: "memory");
    const uint8_t* base = smem + wave * (D * STEP * 1024) + slot * (STEP * 1024);
    i32x4 av[2][MT], bv[2][WT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const uint8_t* q = base + mt * 2048 + (2 * mt + 1 < MX ? upper : 0);
      av[0][mt] = *reinterpret_cast<const i32x4*>(q + at0);
      av[1][mt] = *reinterpret_cast<const i32x4*>(q + at1);
    }
#pragma unroll
    for (int t = 0; t < WT; ++t) {
      const uint8_t* q = base + MX * 1024 + t * 2048 + (2 * t + 1 < WX ? upper : 0);
      bv[0][t] = *reinterpret_cast<const i32x4*>(q + at0);
      bv[1][t] = *reinterpret_cast<const i32x4*>(q + at1);
    }
    // everything is in registers: the slot is free
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (s + D * kMqWaves < steps) copy_step(s + D * kMqWaves, slot);
#pragma unroll
    for (int t = 0; t < WT; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[t][mt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[0][mt], bv[0][t], acc[t][mt], 0, 0, 0);
    if (s * 128 + 64 < K) {
#pragma unroll
      for (int t = 0; t < WT; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[t][mt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[1][mt], bv[1][t], acc[t][mt], 0, 0, 0);
    }
    slot = slot + 1 == D ? 0 : slot + 1;
  }

  // ---- sums of the waves, [wave][row of a][row of b + 4] (rings and sums share the memory) -------------
  __syncthreads();
  int* red = reinterpret_cast<int*>(smem);
  constexpr int RP = R + 4;
  const int waves = steps < kMqWaves ? steps : kMqWaves;  // that have a sum
  if (wave < waves) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = mt * 16 + 4 * kb + v;
        if (m < M) {
#pragma unroll
          for (int t = 0; t < WT; ++t) red[(wave * M + m) * RP + t * 16 + r] = acc[t][mt][v];
        }
      }
  }
  __syncthreads();
  asm volatile("" : "+v"(sb), "+v"(bias_lo), "+v"(bias_hi));
  const float bias = wide ? __builtin_bit_cast(float, bias_lo | bias_hi << 16)
                     : p.out_dtype == OFQ_F16 ? (float)__builtin_bit_cast(f16, (uint16_t)bias_lo)
                                              : __builtin_bit_cast(float, bias_lo << 16);
  constexpr int kRowsAtOnce = kMqWaves * 64 / R;
  if (tid >= kRowsAtOnce * R || orow >= rows_blk) return;
  for (int m = tid / R; m < M; m += kRowsAtOnce) {
    const int* src = red + m * RP + orow;
    int sum = 0;
    if (waves == kMqWaves) {
#pragma unroll
      for (int w = 0; w < kMqWaves; ++w) sum += src[w * M * RP];
    } else {
      for (int w = 0; w < waves; ++w) sum += src[w * M * RP];
    }
    const float v = (float)sum * (sa * sb);
    const int64_t at = (int64_t)m * N + row0 + orow;
    if (p.out_dtype == OFQ_F16) mq_store<f16>(p, at, v, has_bias, bias);
    else if (p.out_dtype == OFQ_BF16) mq_store<bf16>(p, at, v, has_bias, bias);
    else mq_store<float>(p, at, v, has_bias, bias);
  }
}

template<int MX, int WX>
int launch_stream_inst(hipStream_t st, const uint8_t* a, const uint8_t* b, const MqStreamArgs& p) {
  constexpr int STEP = MX + WX, R = (WX + 1) / 2 * 16;
  size_t lds = (size_t)kMqWaves * mq_depth(STEP) * STEP * 1024;
  const size_t red = (size_t)kMqWaves * p.M * (R + 4) * 4;
  if (red > lds) lds = red;
  auto kern = matmul_quant_stream<MX, WX>;
  static std::atomic<uint64_t> lds_allowed{0};  // devices on which the kernel's LDS limit is raised
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), 160 * 1024, lds_allowed)) return OFQ_ERR_LAUNCH;
  kern<<<(unsigned)((p.N + p.rows_per_block - 1) / p.rows_per_block), kMqWaves * 64, lds, st>>>(a, b, p);
  return ofq_check_launch();
}

template<int MX>
int launch_stream_mx(hipStream_t st, const uint8_t* a, const uint8_t* b, const MqStreamArgs& p) {
  switch ((p.rows_per_block + 7) / 8) {
    case 1: return launch_stream_inst<MX, 1>(st, a, b, p);
    case 2: return launch_stream_inst<MX, 2>(st, a, b, p);
    case 3: return launch_stream_inst<MX, 3>(st, a, b, p);
    case 4: return launch_stream_inst<MX, 4>(st, a, b, p);
    case 5: return launch_stream_inst<MX, 5>(st, a, b, p);
    case 6: return launch_stream_inst<MX, 6>(st, a, b, p);
    case 7:
      if constexpr (MX <= 8) return launch_stream_inst<MX, 7>(st, a, b, p);
      break;
    case 8:
      if constexpr (MX <= 8) return launch_stream_inst<MX, 8>(st, a, b, p);
      break;
    default: break;
  }
  return OFQ_ERR_UNSUPPORTED;
}

int launch_stream(hipStream_t st, const uint8_t* a, const uint8_t* b, const MqStreamArgs& args) {
  MqStreamArgs p = args;
  constexpr int64_t kCUs = 256;
  // one block a CU and round, its rows whole: a block of eight rows at least
  const int64_t most = mq_max_rows(p.M);
  const int64_t rounds = (p.N + kCUs * most - 1) / (kCUs * most);
  p.rows_per_block = (int)((p.N + kCUs * rounds - 1) / (kCUs * rounds));
  if (p.rows_per_block < 8) p.rows_per_block = 8;
  if (p.M <= 8) return launch_stream_mx<1>(st, a, b, p);
  if (p.M <= 16) return launch_stream_mx<2>(st, a, b, p);
  if (p.M <= 32) return launch_stream_mx<4>(st, a, b, p);
  if (p.M <= 48) return launch_stream_mx<6>(st, a, b, p);
  if (p.M <= 64) return launch_stream_mx<8>(st, a, b, p);
  if (p.M <= 80) return launch_stream_mx<10>(st, a, b, p);
  return launch_stream_mx<12>(st, a, b, p);
}

// ---- one row of a: a wave owns whole rows of b -----------------------------------------------
// The matrix core has nothing to add, and the ring, its barrier and its fold cost more than they give (11008 x 4096
// 9.2 us against 9.6).  Here lane l holds bytes [h * 1024 + 16 l, +16) of the row of a in registers (h < H =
// ceil(k / 1024)), a wave walks the rows w, w + NW, .. of the block's share of b with the requests of two rows in
// flight, meets each row with v_dot4_i32_i8 (exact int32) and sums across the lanes; no LDS, no barrier.  Same
// int32 sums and the same epilogue as the other paths, hence the same bits.  Two to four rows of a, which this
// kernel held in registers too, stream faster (2 rows: 4096 x 4096 5.7 -> 5.2 us, 2048 x 8192 6.2 -> 5.2, 4 rows of
// 11008 x 4096 12.1 -> 10.0; weights from HBM).
__device__ __forceinline__ int wave_sum_i32(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
  v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
  v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, false);  // row_half_mirror
  v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, false);  // row_mirror
  return (__builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16))
         + (__builtin_amdgcn_readlane(v, 32) + __builtin_amdgcn_readlane(v, 48));
}

template<typename T, int NW, int H>
__global__ void __launch_bounds__(NW * 64)
matmul_quant_wave_rows(const uint8_t* __restrict__ a, const uint8_t* __restrict__ b,
                       const float* __restrict__ a_scale, const float* __restrict__ b_scale,
                       const typename TT<T>::storage* __restrict__ bias,
                       typename TT<T>::storage* __restrict__ out, int N, int K, int rows_per_block) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = blockIdx.x * rows_per_block;
  int rows_blk = N - row0;
  if (rows_blk > rows_per_block) rows_blk = rows_per_block;
  const int nr = rows_blk > wave ? (rows_blk - wave + NW - 1) / NW : 0;  // rows of this wave
  bool valid[H];
  uint32_t voff[H];
#pragma unroll
  for (int h = 0; h < H; ++h) {
    valid[h] = h * 1024 + lane * 16 < K;
    voff[h] = valid[h] ? (uint32_t)(h * 1024 + lane * 16) : 0u;
  }
  const uint8_t* bblk = b + (int64_t)row0 * K;
  i32x4 wq[2][H];
  auto issue = [&](int i, int buf) {
    const bool live = i < nr;  // the same for every lane
    const uint8_t* rowp = bblk + (size_t)(live ? wave + i * NW : 0) * K;
#pragma unroll
    for (int h = 0; h < H; ++h) {
      wq[buf][h] = __builtin_nontemporal_load(
          reinterpret_cast<const i32x4*>(rowp + (live ? voff[h] : 0u)));
    }
  };
  // a first (it comes from L2 and every row of b needs it), then two rows of b
  i32x4 av[H];
#pragma unroll
  for (int h = 0; h < H; ++h) av[h] = *reinterpret_cast<const i32x4*>(a + voff[h]);
  issue(0, 0);
  issue(1, 1);
  const float sa = a_scale[0];
  auto finish = [&](int i, int buf) {
    const int n = row0 + wave + i * NW;
    const float sb = b_scale[n];
    float bv = 0.f;
    if (bias != nullptr) bv = TT<T>::load(bias + n);
    int acc = 0;
#pragma unroll
    for (int h = 0; h < H; ++h) {
      int part = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) part = __builtin_amdgcn_sdot4(av[h][j], wq[buf][h][j], part, false);
      acc += valid[h] ? part : 0;
    }
    const int sum = wave_sum_i32(acc);
    if (lane == 0) {
      float v = (float)sum * (sa * sb);
      if (bias != nullptr) v = v + bv;
      TT<T>::store(out + n, v);
    }
  };
  for (int i = 0; i < nr; i += 2) {
    finish(i, 0);
    issue(i + 2, 0);
    if (i + 1 < nr) finish(i + 1, 1);
    issue(i + 3, 1);
  }
}

template<typename T, int H>
int launch_wave_rows_inst(hipStream_t st, const uint8_t* a, const uint8_t* b, const float* a_scale,
                          const float* b_scale, const void* bias, void* out, int64_t n, int64_t k) {
  typedef typename TT<T>::storage S;
  constexpr int NW = 16;
  // 16 waves per CU, twice as many blocks from 128 rows per block on; a wave then walks its rows
  // two ahead
  int64_t grid = 256;
  if ((n + grid - 1) / grid >= 128) grid *= 2;
  int rpb = (int)((n + grid - 1) / grid);
  if (rpb < NW) rpb = NW;
  grid = (n + rpb - 1) / rpb;
  matmul_quant_wave_rows<T, NW, H><<<(unsigned)grid, NW * 64, 0, st>>>(
      a, b, a_scale, b_scale, static_cast<const S*>(bias), static_cast<S*>(out), (int)n, (int)k, rpb);
  return ofq_check_launch();
}

// one row of up to 8192 elements (it is held in registers)
template<typename T>
int launch_wave_rows(hipStream_t st, const uint8_t* a, const uint8_t* b, const float* a_scale,
                     const float* b_scale, const void* bias, void* out, int64_t n, int64_t k) {
#define OFQ_WR(HV) \
  case HV: return launch_wave_rows_inst<T, HV>(st, a, b, a_scale, b_scale, bias, out, n, k);
  switch ((k + 1023) / 1024) {
    OFQ_WR(1) OFQ_WR(2) OFQ_WR(3) OFQ_WR(4) OFQ_WR(5) OFQ_WR(6) OFQ_WR(7) OFQ_WR(8)
    default: return OFQ_ERR_UNSUPPORTED;
  }
#undef OFQ_WR
}

template<typename T>
int launch_part(hipStream_t st, const uint8_t* a, const uint8_t* b, const float* a_scale,
                const float* b_scale, const void* bias, void* out, int m, int64_t n, int64_t k) {
  if (m == 1 && k <= 8192) return launch_wave_rows<T>(st, a, b, a_scale, b_scale, bias, out, n, k);
  return launch_stream(st, a, b, MqStreamArgs{a_scale, b_scale, bias, out, TT<T>::dtype, m, (int)n, (int)k, 0});
}

}  // namespace

// Expected time in us of 65 rows of a and more (fitted to 1058 random products, within 11 % for 90 of 100): the start, a
// part for every round of blocks, its k-tiles of 128 bytes with the rows of a and of b that a block takes in,
// and the outputs.
double matmul_quant_rows_us(int64_t m, int64_t n, int64_t k) {
  static const double c[2][5] = {{2.06, 1.68, 0.101, 0.264, 2.26}, {1.80, 1.70, 0.145, 0.317, 2.13}};
  const double* f = c[k % 128 != 0];
  const int64_t rounds = (n + 256 * mq_max_rows((int)m) - 1) / (256 * mq_max_rows((int)m));
  const double rows = std::max<int64_t>(8, (n + 256 * rounds - 1) / (256 * rounds));
  const double share = std::min(1.0, std::ceil((double)n / rows) / 256);
  const double kt = (double)((k + 127) / 128) * (double)rounds;
  return f[0] + f[1] * (double)rounds + kt * (f[2] * (m <= 80 ? 0.80 : 0.96) + f[3] * share * rows / 48)
         + f[4] * 1e-6 * (double)m * (double)n;
}

bool matmul_quant_rows_supported(int64_t m, int64_t n, int64_t k) {
  return m >= 1 && m <= kMqMaxM && n >= 1 && k % 64 == 0 && k <= (1 << 24) && n <= 0x7FFFFFFF - 64;
}

// a [m,k], b [n,k] int8, m <= 96
int launch_matmul_quant_rows(hipStream_t st, const void* a, const void* b, const float* a_scale,
                             const float* b_scale, const void* bias, void* out, int out_dtype,
                             int64_t m, int64_t n, int64_t k) {
  const uint8_t* ap = static_cast<const uint8_t*>(a);
  const uint8_t* bp = static_cast<const uint8_t*>(b);
  switch (out_dtype) {
    case OFQ_F16: return launch_part<f16>(st, ap, bp, a_scale, b_scale, bias, out, (int)m, n, k);
    case OFQ_BF16: return launch_part<bf16>(st, ap, bp, a_scale, b_scale, bias, out, (int)m, n, k);
    case OFQ_F32: return launch_part<float>(st, ap, bp, a_scale, b_scale, bias, out, (int)m, n, k);
    default: return OFQ_ERR_BAD_DTYPE;
  }
}

}  // namespace ofq
