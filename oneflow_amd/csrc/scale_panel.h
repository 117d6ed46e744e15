// Scales (and zeros) of a block's weight rows -> LDS, for kernels whose lanes need them by row.
#pragma once

#include "ofq_device.h"

namespace ofq {
namespace {

template<int U, int NT, bool ZERO, bool GROUP_MAJOR>
__device__ __forceinline__ void copy_scale_panel_u(const uint16_t* __restrict__ scale,
                                                   const uint16_t* __restrict__ zero, int G, int total,
                                                   int row_limit, int groups, int pitch, uint16_t* sl,
                                                   uint16_t* zl, int tid) {
  for (int e0 = tid; e0 < total; e0 += NT * U) {
    uint16_t sv[U], zv[U];
    int at[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = e0 + u * NT < total ? e0 + u * NT : e0;
      int row = e / groups;
      const int g = e - row * groups;
      at[u] = GROUP_MAJOR ? g * pitch + row : row * pitch + g;
      row = row < row_limit ? row : row_limit - 1;
      sv[u] = scale[(int64_t)row * G + g];
      if (ZERO) zv[u] = zero[(int64_t)row * G + g];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      sl[at[u]] = sv[u];
      if (ZERO) zl[at[u]] = zv[u];
    }
  }
}

// rows x groups 16-bit values, row r at scale + r * G (rows past row_limit repeat the last one), to
// sl[g * pitch + r] (GROUP_MAJOR) or sl[r * pitch + g].  A thread's requests go out together, eight
// where it has that many: one at a time, each waits for memory.
template<int NT, bool ZERO, bool GROUP_MAJOR>
__device__ __forceinline__ void copy_scale_panel(const uint16_t* __restrict__ scale,
                                                 const uint16_t* __restrict__ zero, int G, int rows,
                                                 int row_limit, int groups, int pitch, uint16_t* sl,
                                                 uint16_t* zl, int tid) {
  const int total = rows * groups;
  if (total > 2 * NT) {
    copy_scale_panel_u<8, NT, ZERO, GROUP_MAJOR>(scale, zero, G, total, row_limit, groups, pitch, sl, zl,
                                                 tid);
  } else {
    copy_scale_panel_u<2, NT, ZERO, GROUP_MAJOR>(scale, zero, G, total, row_limit, groups, pitch, sl, zl,
                                                 tid);
  }
}

}  // namespace
}  // namespace ofq
