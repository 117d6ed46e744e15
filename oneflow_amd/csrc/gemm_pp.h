// Copy-fed MFMA GEMM whose two groups of waves take turns on the matrix cores: out[m, n] =
// a[m, k] b[n, k]^T, both operands as stored (int8, or fp16 / bf16).  Tiles, LDS layout, swizzle and
// epilogue are gemm_core2's (gemm_kernels.h).
#pragma once

#include "gemm_kernels.h"

namespace ofq {
namespace {

// Pieces [LO, HI) of the copies of k-tile kt (rows of a first, then of b; piece j is 64 rows, 8 of
// them by each wave) into a stage.  One lane offset serves every piece: the piece is in the scalar
// base, rows past the matrix repeat its last one by a minimum on the offset.
template<bool RAGGED, int BM, int LO, int HI>
__device__ __forceinline__ void copy_pieces(const uint8_t* __restrict__ a_kt,
                                            const uint8_t* __restrict__ b_kt, uint32_t ld,
                                            uint32_t lane_row_off, uint32_t lane_piece,
                                            uint32_t a_last, uint32_t b_last, bool lane_in_row,
                                            uint8_t* stage, int wave, int lane) {
  const uint32_t lds0 =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)stage + wave * 1024;
#pragma unroll
  for (int j = LO; j < HI; ++j) {
    const bool is_a = j < BM / 64;
    const int jr = is_a ? j : j - BM / 64;
    uint32_t off = lane_row_off + (uint32_t)jr * 64u * ld;
    const uint32_t last = is_a ? a_last : b_last;
    off = (off < last ? off : last) + lane_piece;
    if (!RAGGED || lane_in_row) {
      async_copy16_at(is_a ? a_kt : b_kt, off, lds0 + j * 8192);
    } else {
      *reinterpret_cast<u32x4*>(stage + wave * 1024 + j * 8192 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
    }
  }
}

// gemm_core2 keeps its eight waves in step: after the barrier of a k-tile both waves of a SIMD fetch
// fragments while the matrix cores idle.  Here waves 0-3 and 4-7 (one of each on every SIMD) are one
// slot apart: in a slot one group fetches the fragments of a k-step and requests copies while the
// other multiplies, and a barrier swaps the roles.
//
// Slots of group 0 in a k-tile: fetch 0, multiply 0, fetch 1, ... multiply 3; group 1 does the same one
// slot later.  The other stage is free once group 1 has fetched the last k-steps of
// the tile before, i.e. in the slot in which group 0 fetches first; copies are requested in the fetch
// slots from there on, and each wave waits for its own before the barrier that opens the next tile
// (group 0 in its last multiplying slot, group 1 in its last fetching one).
//
// What bounds it: the clock that the chip gives matrix instructions on random operands, then the copies.
// 8192 x 11008 x 4096 on 256 x 384 tiles, launches in a row: int8 341 us (2.17 POP/s; gemm_core2 371), bf16
// 572 us (1.29 PFLOP/s; 646); 2048 rows: int8 87 us (89), bf16 146 (150); among a pass's other kernels 374
// and 163.  Taken apart when it was built, in runs whose whole took int8 314 us and bf16 550: groups in
// step 365, no copies 290 / 454, no epilogue 277 / 526, no fetches - / 525, neither fetches nor copies 270.
// In the same runs, and not taken: waves of 128 x 96 (fewer LDS reads: 314 / 563), copies spread over more
// slots (312 / 558) or requested before the fetches (320 / 564), rows of 64 bytes in a ring of four stages
// (three in flight: 355 / 621, half lines cost more than the distance gives), non-temporal stores (1.5 %).
template<class MF, bool RAGGED, class EP, int BN>
__global__ void __launch_bounds__(512)
gemm_pp(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, int64_t ld,
        typename EP::Params ep, int M, int N, int KT, int m_tiles, int n_tiles) {
  constexpr int BM = 256;
  constexpr int TM = 2, TN = BN / 64;  // waves 4 x 2, 64 x BN/2 each
  constexpr int kABytes = BM * kStageRow;
  constexpr int kStage = (BM + BN) * kStageRow;
  constexpr int kPieces = (BM + BN) / 64;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

  // an XCD takes consecutive tiles; within them 8 row tiles share a column of b, so that the 32
  // blocks an XCD runs at a time read 8 row tiles of a and 4 column tiles of b through its L2
  int mt, nt;
  {
    const int nblocks = m_tiles * n_tiles;
    const int b = blockIdx.x;
    const int xcd = b & 7, idx = b >> 3;
    const int per = nblocks >> 3, rem = nblocks & 7;
    const int logical = xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
    constexpr int kPanel = 8;
    const int panel = logical / (kPanel * n_tiles);
    const int in_panel = logical - panel * kPanel * n_tiles;
    const int left = m_tiles - panel * kPanel;
    const int height = left < kPanel ? left : kPanel;
    nt = in_panel / height;
    mt = panel * kPanel + in_panel - nt * height;
  }
  const int m0 = mt * BM, n0 = nt * BN;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool late = wave >= 4;  // the group that runs one slot behind
  const int wm0 = (wave >> 1) * 64;
  const int wn0 = (wave & 1) * (BN / 2);

  typename MF::Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;

  const uint8_t* a0 = A + (int64_t)m0 * ld;
  const uint8_t* b0 = B + (int64_t)n0 * ld;
  const uint32_t a_last = (uint32_t)((M - m0 < BM ? M - m0 : BM) - 1) * (uint32_t)ld;
  const uint32_t b_last = (uint32_t)((N - n0 < BN ? N - n0 : BN) - 1) * (uint32_t)ld;
  const uint32_t row_off = (uint32_t)(wave * 8 + (lane >> 3)) * (uint32_t)ld;
  const uint32_t piece = (uint32_t)(((lane & 7) ^ swizzle_key(wave * 8 + (lane >> 3))) * 16);

  const int frag_row = lane & 31;
  const int key = swizzle_key(frag_row);
  const int half = lane >> 5;
  const int a_base = (wm0 + frag_row) * kStageRow;
  const int b_base = kABytes + (wn0 + frag_row) * kStageRow;

#define OFQ_PP_COPY(LO, HI, T)                                                                     \
  copy_pieces<RAGGED, BM, LO, HI>(a0 + (int64_t)(T) * kStageRow, b0 + (int64_t)(T) * kStageRow,      \
                                  (uint32_t)ld, row_off, piece, a_last, b_last,                      \
                                  (T) * kStageRow + (int)piece < (int)ld, lds + ((T) & 1) * kStage,  \
                                  wave, lane)
  OFQ_PP_COPY(0, kPieces, 0);
  wait_vmem_all();
  __syncthreads();
  if (late) __builtin_amdgcn_s_barrier();

  for (int kt = 0; kt < KT; ++kt) {
    const uint8_t* cur = lds + (kt & 1) * kStage;
    const bool more = kt + 1 < KT;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      // ---- fetch --------------------------------------------------------------------------------
      u32x4 af[TM], bf[TN];
      const int off = ((2 * p + half) ^ key) << 4;
#pragma unroll
      for (int i = 0; i < TM; ++i)
        af[i] = *reinterpret_cast<const u32x4*>(cur + a_base + i * 32 * kStageRow + off);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        bf[j] = *reinterpret_cast<const u32x4*>(cur + b_base + j * 32 * kStageRow + off);
      if (more) {
        if (p == 0) OFQ_PP_COPY(0, kPieces / 2, kt + 1);
        if (p == 1) OFQ_PP_COPY(kPieces / 2, kPieces, kt + 1);
      }
      if (p == 3 && late) wait_vmem_all();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      // ---- multiply -----------------------------------------------------------------------------
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = MF::mma(bf[j], af[i], acc[i][j]);
      __builtin_amdgcn_s_setprio(0);
      if (p == 3 && !late) wait_vmem_all();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      // (the last barrier of the late group would have no partner: both groups pass as many)
      if (p < 3 || more || !late) __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#undef OFQ_PP_COPY
  // group 0 is past the barrier behind the late group's last fetch: nobody reads the stages any more
  store_wave_tile<MF, EP, TM, TN, 8, 2 * kStage>(ep, acc, lds, m0 + wm0, n0 + wn0, M, N, wave, lane);
}

template<class MF, bool RAGGED, class EP, int BN>
int launch_pp_tile(hipStream_t st, const void* a, const void* b, int64_t row_bytes,
                   const typename EP::Params& ep, int64_t M, int64_t N) {
  const int m_tiles = (int)((M + 255) / 256);
  const int n_tiles = (int)((N + BN - 1) / BN);
  constexpr int kLds = 2 * (256 + BN) * kStageRow;
  auto kern = gemm_pp<MF, RAGGED, EP, BN>;
  static std::atomic<uint64_t> lds_allowed{0};  // devices on which the kernel's LDS limit is raised
  if (!ofq_allow_dynamic_lds(reinterpret_cast<const void*>(kern), kLds, lds_allowed)) return OFQ_ERR_LAUNCH;
  // the copies address a tile's rows with 32-bit offsets from its first row
  if (row_bytes * (int64_t)(BN > 256 ? BN : 256) >= ((int64_t)1 << 32)) return OFQ_ERR_UNSUPPORTED;
  const int64_t KT = (row_bytes + kStageRow - 1) / kStageRow;
  if (KT < 1 || row_bytes > 0x7FFFFFFF - kStageRow) return OFQ_ERR_UNSUPPORTED;
  kern<<<m_tiles * n_tiles, 512, kLds, st>>>(static_cast<const uint8_t*>(a),
                                             static_cast<const uint8_t*>(b), row_bytes, ep, (int)M,
                                             (int)N, (int)KT, m_tiles, n_tiles);
  return ofq_check_launch();
}

// width: what pick_copy_tile says.  This kernel against gemm_core2, time over time in the mean of 1200 random
// problems (m to 8192, n to 32000, k to 14336; p. 95 is 2 to 5 % above the mean):
//              rows of whole k-tiles: up to 16, 48, more    ragged rows: the same
//   int8  192    0.99  0.99  0.98                           1.01  1.02  1.05
//         256    0.98  0.97  0.93                           0.99  1.00  1.01
//         384    0.98  0.97  0.94                           0.94  0.86  0.85
//   fp16  192    0.99  0.98  0.97                           1.03  1.05  1.07
//         256    0.99  0.97  0.95                           1.00  1.01  1.03
//         384    0.99  0.97  0.95                           0.93  0.85  0.82
//   bf16  192    1.00  0.99  0.96                           1.03  1.04  1.06
//         256    0.99  0.96  0.94                           1.00  1.01  1.05
//         384    0.98  0.97  0.95                           0.92  0.85  0.81
// So ragged rows at 192 columns, and at 256 in 16 bits, stay with gemm_core2 (whose kernel for ragged rows
// runs out of registers at 384 columns and nowhere else).  So do tiles of 128 columns: a slot of four
// matrix instructions is too short for the fetch beside it (1100 x 4096 x 4096: int8 33.3 us there, 35.2
// here, bf16 57.3 and 60.9).
template<class MF, class EP>
int launch_pp(hipStream_t st, const void* a, const void* b, int64_t row_bytes,
              const typename EP::Params& ep, int64_t M, int64_t N, int width) {
  constexpr bool kInt8 = std::is_same<MF, MfmaI8>::value;
  const bool ragged = row_bytes % kStageRow != 0;
  if (width == 384) {
    return ragged ? launch_pp_tile<MF, true, EP, 384>(st, a, b, row_bytes, ep, M, N)
                  : launch_pp_tile<MF, false, EP, 384>(st, a, b, row_bytes, ep, M, N);
  }
  if (width == 256) {
    if (!ragged) return launch_pp_tile<MF, false, EP, 256>(st, a, b, row_bytes, ep, M, N);
    if constexpr (kInt8) return launch_pp_tile<MF, true, EP, 256>(st, a, b, row_bytes, ep, M, N);
  }
  if (width == 192 && !ragged) return launch_pp_tile<MF, false, EP, 192>(st, a, b, row_bytes, ep, M, N);
  return OFQ_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace ofq
