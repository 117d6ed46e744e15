// GEMM on two copied operands, out = A[m, k] B[n, k]^T with rows of 128-byte k-tiles (int8, and 16-bit behind a
// converted weight), for products whose blocks are too few or whose tiles are too small to hide a copy behind the
// products of one k-tile: NSTAGE LDS stages, NSTAGE - 1 k-tiles of copies under way, one barrier a k-tile.
//
// What bounds it: what a CU takes in, 53 to 60 bytes per ns whatever the tile, the stages and the blocks beside it (a
// bare loop of such copies, 8 rows x 128 bytes, reaches 62 with 4 waves, 80 with 8 and 90 with 16; of whole KBs 140): 64 x 64
// tiles 0.30 us a k-tile of 16 KB, 128 x 64 0.41 (24 KB), 128 x 128 0.60 (32 KB), 256 x 128 0.85 (48 KB), where
// one k-tile under way took 0.8, 0.95 and 1.15 us for 64, 128 and 256 rows.  Five stages of 64 x 64 are what the
// latency needs (three: 256 x 4096 x 4096 16.6 us, five 13.0, ten 14.3).  Eight waves of 32 x 64 results beat four of
// 64 x 64 (512 x 4096 x 4096 22.3 against 24.2 us) though they read LDS half as often again; copies between
// the products and not ahead of them give 2 to 10 %, copies that do not order the LDS reads around them 1 to 3 %.
// Blocks that start at different k-tiles are no faster: the L2 channels are not what collides.
#pragma once

#include "gemm_kernels.h"

namespace ofq {
namespace {

// all but the copies of the youngest n <= MOST k-tiles of OPS copies have landed
template<int OPS, int MOST>
__device__ __forceinline__ void wait_tiles(int n) {
  static_assert(OPS * MOST < 64, "vmcnt is a 6-bit counter");
  if constexpr (MOST == 0) {
    wait_vmem_all();
  } else {
    if (n >= MOST) wait_vmem_le<OPS * MOST>();
    else wait_tiles<OPS, MOST - 1>(n);
  }
}

template<class MF, bool RAGGED, class EP, int BM, int BN, int WM, int WN, int NSTAGE>
__global__ void __launch_bounds__(WM * WN * 64)
gemm_deep(const uint8_t* __restrict__ A, int64_t lda, BCopyParams bp, typename EP::Params ep, int M, int N,
          int KT_total, int kt_split, int m_tiles, int n_tiles) {
  constexpr int NWAVES = WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  constexpr int kABytes = BM * kStageRow;
  constexpr int kStage = (BM + BN) * kStageRow;
  constexpr int D = NSTAGE - 1;
  static_assert(NSTAGE >= 3 && BM % (8 * NWAVES) == 0 && BN % (8 * NWAVES) == 0,
                "every wave has the same number of copies");
  constexpr int kOps = (BM + BN) / (8 * NWAVES);
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

  // slices of K: blockIdx.y owns k-tiles [kt_base, kt_base + KT); tile t below is the block's t-th
  const int kt_base = EP::kSplit ? (int)blockIdx.y * kt_split : 0;
  const int KT = EP::kSplit ? (KT_total - kt_base < kt_split ? KT_total - kt_base : kt_split) : KT_total;
  if (EP::kSplit) ep.out += (int64_t)blockIdx.y * M * N;

  // an XCD takes consecutive tiles: those of one strip of columns share its rows of B in the XCD's L2
  const int nblocks = m_tiles * n_tiles;
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  const int per = nblocks >> 3, rem = nblocks & 7;
  const int logical = xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
  const int m0 = (logical % m_tiles) * BM;
  const int n0 = (logical / m_tiles) * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave / WN) * WTM;
  const int wn0 = (wave % WN) * WTN;

  typename MF::Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;

  // A wave's copies of a k-tile, 8 rows x 128 bytes each, the pieces of a row swizzled for the fragment reads: the
  // first of A's rows, the others of B's; rows past the end re-read the last one.  Past the end of a row (ragged K, its
  // last k-tile) a lane writes zeros of its own.
  constexpr int kAOps = BM / (8 * NWAVES);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  uint32_t off[kOps];
  int piece[kOps];  // its byte in the k-tile
#pragma unroll
  for (int o = 0; o < kOps; ++o) {
    const int row = ((o < kAOps ? o : o - kAOps) * NWAVES + wave) * 8 + (lane >> 3);
    const int last = o < kAOps ? M - 1 - m0 : N - 1 - n0;
    piece[o] = ((lane & 7) ^ swizzle_key(row)) * 16;
    off[o] = (uint32_t)(row < last ? row : last) * (uint32_t)(o < kAOps ? lda : bp.ldb) + (uint32_t)piece[o];
  }
  const uint8_t* const a_rows = A + (int64_t)m0 * lda;
  const uint8_t* const b_rows = bp.b + (int64_t)n0 * bp.ldb;
  auto copy = [&](int t, int stage, int o) {
    const int64_t at = (int64_t)(kt_base + t) * kStageRow;
    const bool is_a = o < kAOps;
    const int to = stage * kStage + (is_a ? 0 : kABytes) + ((is_a ? o : o - kAOps) * NWAVES + wave) * 1024;
    if (!RAGGED || at + piece[o] < lda) {  // (both operands have rows of the same K)
      async_copy16_unordered((is_a ? a_rows : b_rows) + at, off[o], lds0 + (uint32_t)to);
    } else {
      *reinterpret_cast<u32x4*>(lds + to + lane * 16) = u32x4{0u, 0u, 0u, 0u};
    }
  };
  // k-tile t + 1 is complete, everyone's, and everyone has done with k-tile t: what is in flight stays so
  // (__syncthreads would wait for it)
  auto next_tile = [&](int t) {
    wait_tiles<kOps, D - 1>(KT - 2 - t);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
#pragma unroll
  for (int t = 0; t < D; ++t)
    if (t < KT) {
#pragma unroll
      for (int o = 0; o < kOps; ++o) copy(t, t, o);
    }
  next_tile(-1);

  // fragments: row = i * 32 + lane % 32 of the wave's rows, piece 2 ks + lane / 32 at its place ^ key(row), which
  // depends on the lane alone (tile origins are multiples of 16)
  const int frag_row = lane & 31;
  const int key = swizzle_key(frag_row);
  const int half = lane >> 5;
  int frag_off[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) frag_off[ks] = ((2 * ks + half) ^ key) << 4;

  int cur = 0, fill = D;  // stages of k-tile kt and of k-tile kt + D
  for (int kt = 0; kt < KT; ++kt) {
    const bool more = kt + D < KT;
    const uint8_t* a_base = lds + cur * kStage + (wm0 + frag_row) * kStageRow;
    const uint8_t* b_base = lds + cur * kStage + kABytes + (wn0 + frag_row) * kStageRow;
    u32x4 af[2][TM], bf[2][TN];
    auto fetch = [&](int ks, int set) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
        af[set][i] = *reinterpret_cast<const u32x4*>(a_base + i * 32 * kStageRow + frag_off[ks]);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        bf[set][j] = *reinterpret_cast<const u32x4*>(b_base + j * 32 * kStageRow + frag_off[ks]);
    };
    fetch(0, 0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks < 3) fetch(ks + 1, (ks + 1) & 1);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = MF::mma(bf[ks & 1][j], af[ks & 1][i], acc[i][j]);
      // the copies of k-tile kt + D a few at a time: a wave that issues them all at once waits for the address unit
      // before its first product
      if (more) {
#pragma unroll
        for (int o = 0; o < kOps; ++o)
          if (o * 4 / kOps == ks) copy(kt + D, fill, o);
      }
    }
    next_tile(kt);
    cur = cur + 1 == NSTAGE ? 0 : cur + 1;
    fill = fill + 1 == NSTAGE ? 0 : fill + 1;
  }
  // all waves passed the last barrier, no copy is under way
  store_wave_tile<MF, EP, TM, TN, NWAVES, NSTAGE * kStage>(ep, acc, lds, m0 + wm0, n0 + wn0, M, N, wave, lane);
}

template<class MF, bool RAGGED, class EP, int BM, int BN, int WM, int WN, int NSTAGE>
int launch_deep(hipStream_t st, const void* A, int64_t lda, const BCopyParams& bp, const typename EP::Params& ep,
                int64_t M, int64_t N, int64_t KT, int splits = 1) {
  const int m_tiles = (int)((M + BM - 1) / BM);
  const int n_tiles = (int)((N + BN - 1) / BN);
  const size_t lds_bytes = NSTAGE * (size_t)(BM + BN) * kStageRow;
  auto kern = gemm_deep<MF, RAGGED, EP, BM, BN, WM, WN, NSTAGE>;
  static std::atomic<uint64_t> lds_allowed{0};  // devices on which the kernel's LDS limit is raised
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), (int)lds_bytes, lds_allowed)) return OFQ_ERR_LAUNCH;
  if (splits < 1 || (splits > 1 && !EP::kSplit)) return OFQ_ERR_UNSUPPORTED;
  // the copies address a tile's rows with 32-bit offsets from its first row
  if (lda * (BM < M ? BM : M) >= ((int64_t)1 << 32) || bp.ldb * (BN < N ? BN : N) >= ((int64_t)1 << 32)) {
    return OFQ_ERR_UNSUPPORTED;
  }
  const int kt_split = (int)((KT + splits - 1) / splits);
  if ((int64_t)kt_split * (splits - 1) >= KT) return OFQ_ERR_UNSUPPORTED;  // an empty slice
  kern<<<dim3(m_tiles * n_tiles, splits), WM * WN * 64, lds_bytes, st>>>(
      static_cast<const uint8_t*>(A), lda, bp, ep, (int)M, (int)N, (int)KT, kt_split, m_tiles, n_tiles);
  return ofq_check_launch();
}

}  // namespace
}  // namespace ofq
