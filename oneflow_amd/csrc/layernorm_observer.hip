// fused_layer_norm_min_max_observer for gfx950: LayerNorm over the last axis fused with a
// per-tensor symmetric min/max observer of the normalised output.
//
// LayerNorm arithmetic (oneflow/core/cuda/layer_norm.cuh:212-233,377-380 and the affine store of
// oneflow/user/kernels/layer_norm_gpu_kernel.cu:40-70): statistics in fp32,
// var = max(M2/n, 0), inv = rsqrt(var + eps); the normalised value is rounded to T first and the
// affine `* gamma + beta` is then carried out in T (two more roundings).
// Observer (oneflow/user/kernels/min_max_observer_kernel.cu:117-131): scale = absmax / (2^(b-1)-1).
// With SKIP the normalised input is that of skip_layer_norm
// (oneflow/user/kernels/skip_layer_norm_kernel.cu:36-67): (x + bias[c]) + skip * T(alpha), every
// operation rounded to T, an absent bias or skip entering as zero.
//
// Rows of up to 4096 elements: one WAVE per row.  The row is read from HBM once (128-bit loads,
// 1 KB per wave instruction) and kept in registers for the three uses (sum, squared deviations,
// normalise); the reductions are cross-lane only, so no barrier and no LDS is involved and the
// waves of a CU drift apart, which overlaps one wave's loads with another's stores.  Longer rows
// use one block per row; up to 8 rows of a 16-bit type share one block, which needs no second launch
// (ln_quant_rows).  The absmax of the stored values goes to the workspace (one float per
// wave or per row) and a second launch of one block folds them and divides.
#include <atomic>
#include <type_traits>
#include "ofq_device.h"

// Scratch of the entry point that allocates nothing (ofq_fused_layer_norm_min_max_observer_static):
// one partial absmax per row or wave, the role the caller's workspace plays in the other entry
// points.  Every device the library runs on holds its own copy until the process ends.  In host
// code the name below is only a handle for hipGetSymbolAddress; the device address it yields is
// what kernels and copies are given.
#define OFQ_LN_STATIC_MAX_ROWS 65536
static __device__ __align__(256) float scratch[OFQ_LN_STATIC_MAX_ROWS];

namespace ofq {
namespace {

constexpr int kLnBlock = 256;

template<typename T>
struct Pack8 {
  typename TT<T>::storage v[8];
};

template<typename T>
__device__ __forceinline__ void load8(const typename TT<T>::storage* p, float* f) {
  typedef typename TT<T>::storage S;
  S tmp[8];
  if (sizeof(S) == 2) {
    *reinterpret_cast<u32x4*>(tmp) = *reinterpret_cast<const u32x4*>(p);
  } else {
    reinterpret_cast<u32x4*>(tmp)[0] = reinterpret_cast<const u32x4*>(p)[0];
    reinterpret_cast<u32x4*>(tmp)[1] = reinterpret_cast<const u32x4*>(p)[1];
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = TT<T>::load(&tmp[e]);
}

template<typename T>
__device__ __forceinline__ void store8(typename TT<T>::storage* p, const float* f) {
  typedef typename TT<T>::storage S;
  S tmp[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) TT<T>::store(&tmp[e], f[e]);
  if (sizeof(S) == 2) {
    *reinterpret_cast<u32x4*>(p) = *reinterpret_cast<const u32x4*>(tmp);
  } else {
    reinterpret_cast<u32x4*>(p)[0] = reinterpret_cast<const u32x4*>(tmp)[0];
    reinterpret_cast<u32x4*>(p)[1] = reinterpret_cast<const u32x4*>(tmp)[1];
  }
}

// the residual inputs of skip_layer_norm; alpha already rounded to T
template<typename T>
struct SkipArgs {
  const typename TT<T>::storage* bias;  // [cols] or null
  const typename TT<T>::storage* skip;  // [rows, cols] or null
  float alpha;
};

// T((x - mean) * inv) as the reference forms it: the fp32 product, rounded to fp32, is narrowed
// to T (layer_norm.cuh stores through static_cast).  The empty asm keeps the two roundings
// apart: fused into v_fma_mixlo_f16 the product would be rounded to fp16 once, which differs in
// about one element of 30000.
template<typename T>
__device__ __forceinline__ float normalised(float d, float inv) {
  float p = d * inv;
  if constexpr (TT<T>::dtype == OFQ_F16) asm volatile("" : "+v"(p));
  return TT<T>::round(p);
}

template<typename T>
__device__ __forceinline__ float skip_sum(float x, float b, float s, float alpha) {
  return TT<T>::round(TT<T>::round(x + b) + TT<T>::round(s * alpha));
}

// EXACT statistics: the row sum and the squared deviations from the unrounded mean are taken in
// fp64 (a sum of fp16 / bf16 values of ordinary range is exact there in any order, the squares
// carry errors of 1e-16), and mean and inv are each rounded once to the fp32 values the
// normalisation uses -- the correctly rounded statistics of the row, independent of the order of
// summation.  The fp32 statistics (the default) depend on that order in the last bit, as the
// reference's own do.  The cost is three fp64 operations per element and pass.
__device__ __forceinline__ float exact_inv(double m2, double n, double eps) {
  double var = m2 / n;
  if (var < 0.0) var = 0.0;
  return (float)(1.0 / __builtin_sqrt(var + eps));
}

// NP = packs of 8 elements each lane caches; cols <= kLnBlock * 8 * NP and 8 | cols.
template<typename T, int NP, bool SKIP, bool EXACT>
__global__ void __launch_bounds__(kLnBlock)
ln_observer_rows(const typename TT<T>::storage* __restrict__ x,
                 const typename TT<T>::storage* __restrict__ gamma,
                 const typename TT<T>::storage* __restrict__ beta,
                 typename TT<T>::storage* __restrict__ y, float* __restrict__ row_absmax,
                 int64_t cols, double eps64, SkipArgs<T> sk) {
  __shared__ float smem[kLnBlock / kWave];
  __shared__ double smem64[EXACT ? kLnBlock / kWave : 1];
  const float eps = (float)eps64;
  const int64_t row = blockIdx.x;
  const typename TT<T>::storage* xr = x + row * cols;
  typename TT<T>::storage* yr = y + row * cols;
  const int npacks = (int)(cols / 8);
  float v[NP][8];
  float sum = 0.0f;
  double sum64 = 0.0;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = threadIdx.x + i * kLnBlock;
    if (p < npacks) {
      load8<T>(xr + (int64_t)p * 8, v[i]);
      if (SKIP) {
        float bb[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        float ss[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (sk.bias) load8<T>(sk.bias + (int64_t)p * 8, bb);
        if (sk.skip) load8<T>(sk.skip + row * cols + (int64_t)p * 8, ss);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = skip_sum<T>(v[i][e], bb[e], ss[e], sk.alpha);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (EXACT) sum64 += (double)v[i][e];
        else sum += v[i][e];
      }
    }
  }
  float mean, inv;
  if constexpr (EXACT) {
    sum64 = block_reduce(sum64, OpSum(), smem64);
    const double mean64 = sum64 / (double)cols;
    double q = 0.0;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int p = threadIdx.x + i * kLnBlock;
      if (p < npacks) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const double d = (double)v[i][e] - mean64;
          q = __builtin_fma(d, d, q);
        }
      }
    }
    q = block_reduce(q, OpSum(), smem64);
    mean = (float)mean64;
    inv = exact_inv(q, (double)cols, eps64);
  } else {
    sum = block_reduce(sum, OpSum(), smem);
    mean = sum / (float)cols;
    float m2 = 0.0f;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int p = threadIdx.x + i * kLnBlock;
      if (p < npacks) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = v[i][e] - mean;
          m2 = __builtin_fmaf(d, d, m2);
        }
      }
    }
    m2 = block_reduce(m2, OpSum(), smem);
    const float var = fmaxf(m2 / (float)cols, 0.0f);
    inv = 1.0f / __builtin_sqrtf(var + eps);
  }
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = threadIdx.x + i * kLnBlock;
    if (p < npacks) {
      float g[8], b[8], o[8];
      if (gamma) load8<T>(gamma + (int64_t)p * 8, g);
      if (beta) load8<T>(beta + (int64_t)p * 8, b);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float t = normalised<T>(v[i][e] - mean, inv);
        if (gamma) t = TT<T>::round(t * g[e]);
        if (beta) t = TT<T>::round(t + b[e]);
        else if (gamma) t = t + 0.0f;  // the reference adds its default beta 0: -0 becomes +0
        o[e] = t;
        amax = fmaxf(amax, fabsf(t));
      }
      store8<T>(yr + (int64_t)p * 8, o);
    }
  }
  amax = block_reduce(amax, OpMax(), smem);
  if (threadIdx.x == 0) row_absmax[row] = amax;
}

// Raw 8-element packs (16 bytes of fp16/bf16, 32 bytes of fp32) and their widening to fp32.
template<typename T>
struct RawPack {
  u32x4 q[sizeof(typename TT<T>::storage) * 8 / 16];
};
template<typename T>
__device__ __forceinline__ RawPack<T> load_raw(const typename TT<T>::storage* p) {
  RawPack<T> r;
#pragma unroll
  for (int i = 0; i < (int)(sizeof(r.q) / 16); ++i) r.q[i] = reinterpret_cast<const u32x4*>(p)[i];
  return r;
}
// (whole-vector bit casts: element access through the struct member, `r.q[0][w]`, came out of the
// compiler as component 0 for every w)
template<typename T>
__device__ __forceinline__ void widen(const RawPack<T>& r, float* f) {
  if constexpr (TT<T>::dtype == OFQ_F16) {
    const f16x8 h = __builtin_bit_cast(f16x8, r.q[0]);
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = (float)h[i];
  } else if constexpr (TT<T>::dtype == OFQ_BF16) {
    const u16x8 h = __builtin_bit_cast(u16x8, r.q[0]);
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = bf16_to_float(h[i]);
  } else {
    const f32x4 lo = __builtin_bit_cast(f32x4, r.q[0]);
    const f32x4 hi = __builtin_bit_cast(f32x4, r.q[sizeof(r.q) / 16 - 1]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[i] = lo[i];
      f[4 + i] = hi[i];
    }
  }
}

template<typename T>
__device__ __forceinline__ RawPack<T> narrow(const float* f) {
  RawPack<T> r;
  if constexpr (TT<T>::dtype == OFQ_F16) {
    f16x8 h;
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = (f16)f[i];
    r.q[0] = __builtin_bit_cast(u32x4, h);
  } else if constexpr (TT<T>::dtype == OFQ_BF16) {
    u16x8 h;
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = float_to_bf16(f[i]);
    r.q[0] = __builtin_bit_cast(u32x4, h);
  } else {
    r.q[0] = __builtin_bit_cast(u32x4, f32x4{f[0], f[1], f[2], f[3]});
    r.q[sizeof(r.q) / 16 - 1] = __builtin_bit_cast(u32x4, f32x4{f[4], f[5], f[6], f[7]});
  }
  return r;
}

// One wave per row; NP = packs of 8 elements each lane caches: cols <= 64 * 8 * NP and 8 | cols.
// A wave walks rows gw, gw + nwaves, ... and leaves the absmax over all of them in wave_absmax[gw].
// x, gamma and beta are all requested before anything is waited for and stay in registers in
// storage format (half the registers of fp32 for the 16-bit types), so the row's critical path
// holds one memory round trip, not two.
template<typename T, int NP, bool SKIP, bool EXACT>
__global__ void __launch_bounds__(kLnBlock)
ln_observer_wave_rows(const typename TT<T>::storage* __restrict__ x,
                      const typename TT<T>::storage* __restrict__ gamma,
                      const typename TT<T>::storage* __restrict__ beta,
                      typename TT<T>::storage* __restrict__ y, float* __restrict__ wave_absmax,
                      int64_t rows, int64_t cols, double eps64, SkipArgs<T> sk) {
  const float eps = (float)eps64;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t gw = (int64_t)blockIdx.x * (kLnBlock / kWave) + (threadIdx.x >> 6);
  const int64_t nwaves = (int64_t)gridDim.x * (kLnBlock / kWave);
  const int npacks = (int)(cols / 8);
  float amax = 0.0f;
  RawPack<T> gr[NP], br[NP];
  bool first = true;
  for (int64_t row = gw; row < rows; row += nwaves) {
    const typename TT<T>::storage* xr = x + row * cols;
    typename TT<T>::storage* yr = y + row * cols;
    RawPack<T> v[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int p = lane + i * kWave;
      if (p < npacks) v[i] = load_raw<T>(xr + (int64_t)p * 8);
    }
    if (SKIP) {
      // the residual sum, rounded to T, takes the place of x in the registers
      RawPack<T> sr[NP], bb[NP];
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int p = lane + i * kWave;
        if (p < npacks) {
          if (sk.skip) sr[i] = load_raw<T>(sk.skip + row * cols + (int64_t)p * 8);
          if (sk.bias) bb[i] = load_raw<T>(sk.bias + (int64_t)p * 8);
        }
      }
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int p = lane + i * kWave;
        if (p < npacks) {
          float fx[8], fb[8], fs[8], o[8];
          widen<T>(v[i], fx);
#pragma unroll
          for (int e = 0; e < 8; ++e) fb[e] = fs[e] = 0.f;
          if (sk.bias) widen<T>(bb[i], fb);
          if (sk.skip) widen<T>(sr[i], fs);
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = skip_sum<T>(fx[e], fb[e], fs[e], sk.alpha);
          v[i] = narrow<T>(o);
        }
      }
    }
    if (first) {
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int p = lane + i * kWave;
        if (p < npacks) {
          if (gamma) gr[i] = load_raw<T>(gamma + (int64_t)p * 8);
          if (beta) br[i] = load_raw<T>(beta + (int64_t)p * 8);
        }
      }
      first = false;
    }
    float mean, inv;
    if constexpr (EXACT) {
      double sum64 = 0.0;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int p = lane + i * kWave;
        if (p < npacks) {
          float f[8];
          widen<T>(v[i], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) sum64 += (double)f[e];
        }
      }
      sum64 = wave_reduce(sum64, OpSum());
      const double mean64 = sum64 / (double)cols;
      double q = 0.0;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int p = lane + i * kWave;
        if (p < npacks) {
          float f[8];
          widen<T>(v[i], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const double d = (double)f[e] - mean64;
            q = __builtin_fma(d, d, q);
          }
        }
      }
      q = wave_reduce(q, OpSum());
      mean = (float)mean64;
      inv = exact_inv(q, (double)cols, eps64);
    } else {
      float sum = 0.0f;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int p = lane + i * kWave;
        if (p < npacks) {
          // (plain widen-and-add: a chain of v_dot2_f32_f16 on one accumulator came out of the
          // compiler with the same source register in every link)
          float f[8];
          widen<T>(v[i], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) sum += f[e];
        }
      }
      sum = wave_reduce(sum, OpSum());
      mean = sum / (float)cols;
      float m2 = 0.0f;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int p = lane + i * kWave;
        if (p < npacks) {
          float f[8];
          widen<T>(v[i], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float d = f[e] - mean;
            m2 = __builtin_fmaf(d, d, m2);
          }
        }
      }
      m2 = wave_reduce(m2, OpSum());
      const float var = fmaxf(m2 / (float)cols, 0.0f);
      inv = 1.0f / __builtin_sqrtf(var + eps);
    }
    f16x8 amax8 = {(f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f};
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int p = lane + i * kWave;
      if (p < npacks) {
        if constexpr (TT<T>::dtype == OFQ_F16) {
          // the affine in T is native packed fp16 arithmetic: one rounding per multiply and per
          // add, which is what rounding the fp32 result of each step to fp16 gives as well
          float f[8];
          widen<T>(v[i], f);
          f16x8 t;
#pragma unroll
          for (int e = 0; e < 8; ++e) t[e] = (f16)((f[e] - mean) * inv);
          if (gamma) t = t * __builtin_bit_cast(f16x8, gr[i].q[0]);
          if (beta) t = t + __builtin_bit_cast(f16x8, br[i].q[0]);
          else if (gamma) t = t + (f16)0.0f;  // the reference adds its default beta 0: -0 -> +0
          amax8 = __builtin_elementwise_max(amax8, __builtin_elementwise_abs(t));
          *reinterpret_cast<u32x4*>(yr + (int64_t)p * 8) = __builtin_bit_cast(u32x4, t);
        } else {
          float f[8], g[8], b[8], o[8];
          widen<T>(v[i], f);
          if (gamma) widen<T>(gr[i], g);
          if (beta) widen<T>(br[i], b);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            float t = normalised<T>(f[e] - mean, inv);
            if (gamma) t = TT<T>::round(t * g[e]);
            if (beta) t = TT<T>::round(t + b[e]);
            else if (gamma) t = t + 0.0f;  // default beta 0 of the reference: -0 -> +0
            o[e] = t;
            amax = fmaxf(amax, fabsf(t));
          }
          store8<T>(yr + (int64_t)p * 8, o);
        }
      }
    }
    if constexpr (TT<T>::dtype == OFQ_F16) {
#pragma unroll
      for (int e = 0; e < 8; ++e) amax = fmaxf(amax, (float)amax8[e]);
    }
  }
  amax = wave_reduce(amax, OpMax());
  if (lane == 0 && gw < rows) wave_absmax[gw] = amax;
}

// Rows of exactly 512 * NP elements of a 16-bit type, gamma and beta both present, no residual:
// the same one-wave-per-row scheme with nothing conditional inside the row (no partial packs, no
// null checks), the deviations kept in registers between the variance and the normalisation, the
// fp16 row sum formed with packed dot products, and, when a wave walks several rows (LOOP), the
// next row requested before the current one is worked on.  At 2048 x 4096 the general kernel
// spends about 1100 vector instructions per row, this one about half; both are bound by that
// arithmetic once the row has arrived, not by HBM.
// SKIP: the normalised row is (x + bias[c]) + skip * T(alpha) (see the top of the file), formed
// as the row arrives and kept in storage format in place of x; the next row is then not
// requested ahead (LOOP must be false), the registers hold the residual inputs instead.
template<typename T, int NP, bool LOOP, bool SKIP, bool EXACT>
__global__ void __launch_bounds__(kLnBlock)
ln_observer_wave_full(const typename TT<T>::storage* __restrict__ x,
                      const typename TT<T>::storage* __restrict__ gamma,
                      const typename TT<T>::storage* __restrict__ beta,
                      typename TT<T>::storage* __restrict__ y, float* __restrict__ wave_absmax,
                      int64_t rows, double eps64, SkipArgs<T> sk) {
  const float eps = (float)eps64;
  static_assert(sizeof(typename TT<T>::storage) == 2, "16-bit types only");
  static_assert(!(SKIP && LOOP), "the residual variant does not prefetch");
  constexpr int kCols = NP * 512;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t gw = (int64_t)blockIdx.x * (kLnBlock / kWave) + (threadIdx.x >> 6);
  const int64_t nwaves = (int64_t)gridDim.x * (kLnBlock / kWave);
  if (gw >= rows) return;
  u32x4 cur[NP], nxt[LOOP ? NP : 1], gr[NP], br[NP];
  {
    const typename TT<T>::storage* xr = x + gw * kCols + lane * 8;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      cur[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(xr + i * 512));
    }
  }
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    gr[i] = *reinterpret_cast<const u32x4*>(gamma + lane * 8 + i * 512);
    br[i] = *reinterpret_cast<const u32x4*>(beta + lane * 8 + i * 512);
  }
  float amax = 0.0f;
  f16x8 amax8 = {(f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f};
  for (int64_t row = gw; row < rows; row += nwaves) {
    bool more = false;
    if constexpr (LOOP) {
      more = row + nwaves < rows;  // the same for every lane
      if (more) {
        const typename TT<T>::storage* xn = x + (row + nwaves) * kCols + lane * 8;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          nxt[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(xn + i * 512));
        }
      }
    }
    if constexpr (SKIP) {
      if (row != gw) {  // (rows after the wave's first: x was not requested ahead)
        const typename TT<T>::storage* xr2 = x + row * kCols + lane * 8;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          cur[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(xr2 + i * 512));
        }
      }
      u32x4 sr[NP], bb[NP];
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        if (sk.skip) {
          sr[i] = __builtin_nontemporal_load(
              reinterpret_cast<const u32x4*>(sk.skip + row * kCols + lane * 8 + i * 512));
        }
        if (sk.bias) bb[i] = *reinterpret_cast<const u32x4*>(sk.bias + lane * 8 + i * 512);
      }
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        if constexpr (TT<T>::dtype == OFQ_F16) {
          // native packed fp16 arithmetic rounds once per operation, which is what rounding the
          // fp32 result of each operation to fp16 gives as well (an absent input enters as +0)
          f16x8 v = __builtin_bit_cast(f16x8, cur[i]);
          const f16x8 zero8 = {(f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f};
          v = v + (sk.bias ? __builtin_bit_cast(f16x8, bb[i]) : zero8);
          const f16 a = (f16)sk.alpha;
          const f16x8 sa = sk.skip ? __builtin_bit_cast(f16x8, sr[i]) * a : zero8 * a;
          v = v + sa;
          cur[i] = __builtin_bit_cast(u32x4, v);
        } else {
          RawPack<T> xp, sp, bp;
          xp.q[0] = cur[i];
          float fx[8], fb[8], fs[8], o[8];
          widen<T>(xp, fx);
#pragma unroll
          for (int e = 0; e < 8; ++e) fb[e] = fs[e] = 0.f;
          if (sk.bias) { bp.q[0] = bb[i]; widen<T>(bp, fb); }
          if (sk.skip) { sp.q[0] = sr[i]; widen<T>(sp, fs); }
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = skip_sum<T>(fx[e], fb[e], fs[e], sk.alpha);
          cur[i] = narrow<T>(o).q[0];
        }
      }
    }
    float f[NP][8];
    float sum = 0.0f;
    double sum64 = 0.0;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      RawPack<T> rp;
      rp.q[0] = cur[i];
      widen<T>(rp, f[i]);
      if constexpr (EXACT) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sum64 += (double)f[i][e];
      } else if constexpr (TT<T>::dtype == OFQ_F16) {
        // (1, 1) held in a register: with the constant as a literal operand the compiler emits
        // the four dot products of a pack with one and the same source register
        uint32_t ones_bits = 0x3c003c00u;
        asm volatile("" : "+v"(ones_bits));
        const f16x2 ones = __builtin_bit_cast(f16x2, ones_bits);
        // (pairs taken from the whole-vector bit cast: `bit_cast<f16x2>(cur[i][w])` came out of
        // the compiler as word 0 for every w)
        const f16x8 h = __builtin_bit_cast(f16x8, cur[i]);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 0, 1), ones, sum, false);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 2, 3), ones, sum, false);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 4, 5), ones, sum, false);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 6, 7), ones, sum, false);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) sum += f[i][e];
      }
    }
    float mean, inv;
    if constexpr (EXACT) {
      sum64 = wave_reduce(sum64, OpSum());
      const double mean64 = sum64 / (double)kCols;
      mean = (float)mean64;
      double q = 0.0;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const double d = (double)f[i][e] - mean64;
          q = __builtin_fma(d, d, q);
          f[i][e] = f[i][e] - mean;
        }
      }
      q = wave_reduce(q, OpSum());
      inv = exact_inv(q, (double)kCols, eps64);
    } else {
      sum = wave_reduce(sum, OpSum());
      mean = sum / (float)kCols;
      float m2 = 0.0f;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          f[i][e] = f[i][e] - mean;
          m2 = __builtin_fmaf(f[i][e], f[i][e], m2);
        }
      }
      m2 = wave_reduce(m2, OpSum());
      const float var = fmaxf(m2 / (float)kCols, 0.0f);
      inv = 1.0f / __builtin_sqrtf(var + eps);
    }
    typename TT<T>::storage* yr = y + row * kCols + lane * 8;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if constexpr (TT<T>::dtype == OFQ_F16) {
        f16x8 t;
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = (f16)(f[i][e] * inv);
        t = t * __builtin_bit_cast(f16x8, gr[i]);
        t = t + __builtin_bit_cast(f16x8, br[i]);
        // |t| by clearing the sign bits of the four words (elementwise abs of the vector comes
        // out as three instructions per pair)
        const u32x4 tb = __builtin_bit_cast(u32x4, t);
        const u32x4 ab = {tb[0] & 0x7FFF7FFFu, tb[1] & 0x7FFF7FFFu, tb[2] & 0x7FFF7FFFu,
                          tb[3] & 0x7FFF7FFFu};
        amax8 = __builtin_elementwise_max(amax8, __builtin_bit_cast(f16x8, ab));
        *reinterpret_cast<u32x4*>(yr + i * 512) = tb;
      } else {
        RawPack<T> gp, bp;
        gp.q[0] = gr[i];
        bp.q[0] = br[i];
        float g[8], b[8], o[8];
        widen<T>(gp, g);
        widen<T>(bp, b);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float t = normalised<T>(f[i][e], inv);
          t = TT<T>::round(t * g[e]);
          t = TT<T>::round(t + b[e]);
          o[e] = t;
          amax = fmaxf(amax, fabsf(t));
        }
        store8<T>(yr + i * 512, o);
      }
    }
    if constexpr (LOOP) {
      if (more) {
#pragma unroll
        for (int i = 0; i < NP; ++i) cur[i] = nxt[i];
      }
    }
  }
  if constexpr (TT<T>::dtype == OFQ_F16) {
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, (float)amax8[e]);
  }
  amax = wave_reduce(amax, OpMax());
  if (lane == 0) wave_absmax[gw] = amax;
}

// any cols: three passes over the row through L2 (the row was just read, so only the first
// pass touches HBM), scalar accesses.
template<typename T, bool SKIP, bool EXACT>
__global__ void __launch_bounds__(kLnBlock)
ln_observer_rows_generic(const typename TT<T>::storage* __restrict__ x,
                         const typename TT<T>::storage* __restrict__ gamma,
                         const typename TT<T>::storage* __restrict__ beta,
                         typename TT<T>::storage* __restrict__ y, float* __restrict__ row_absmax,
                         int64_t cols, double eps64, SkipArgs<T> sk) {
  __shared__ float smem[kLnBlock / kWave];
  __shared__ double smem64[EXACT ? kLnBlock / kWave : 1];
  const float eps = (float)eps64;
  const int64_t row = blockIdx.x;
  const typename TT<T>::storage* xr = x + row * cols;
  typename TT<T>::storage* yr = y + row * cols;
  auto input = [&](int64_t c) {
    const float xv = TT<T>::load(xr + c);
    if (!SKIP) return xv;
    const float bv = sk.bias ? TT<T>::load(sk.bias + c) : 0.f;
    const float sv = sk.skip ? TT<T>::load(sk.skip + row * cols + c) : 0.f;
    return skip_sum<T>(xv, bv, sv, sk.alpha);
  };
  float mean, inv;
  if constexpr (EXACT) {
    double sum64 = 0.0;
    for (int64_t c = threadIdx.x; c < cols; c += kLnBlock) sum64 += (double)input(c);
    sum64 = block_reduce(sum64, OpSum(), smem64);
    const double mean64 = sum64 / (double)cols;
    double q = 0.0;
    for (int64_t c = threadIdx.x; c < cols; c += kLnBlock) {
      const double d = (double)input(c) - mean64;
      q = __builtin_fma(d, d, q);
    }
    q = block_reduce(q, OpSum(), smem64);
    mean = (float)mean64;
    inv = exact_inv(q, (double)cols, eps64);
  } else {
    float sum = 0.0f;
    for (int64_t c = threadIdx.x; c < cols; c += kLnBlock) sum += input(c);
    sum = block_reduce(sum, OpSum(), smem);
    mean = sum / (float)cols;
    float m2 = 0.0f;
    for (int64_t c = threadIdx.x; c < cols; c += kLnBlock) {
      const float d = input(c) - mean;
      m2 = __builtin_fmaf(d, d, m2);
    }
    m2 = block_reduce(m2, OpSum(), smem);
    const float var = fmaxf(m2 / (float)cols, 0.0f);
    inv = 1.0f / __builtin_sqrtf(var + eps);
  }
  float amax = 0.0f;
  for (int64_t c = threadIdx.x; c < cols; c += kLnBlock) {
    float t = normalised<T>(input(c) - mean, inv);
    if (gamma) t = TT<T>::round(t * TT<T>::load(gamma + c));
    if (beta) t = TT<T>::round(t + TT<T>::load(beta + c));
    else if (gamma) t = t + 0.0f;  // default beta 0 of the reference: -0 -> +0
    TT<T>::store(yr + c, t);
    amax = fmaxf(amax, fabsf(t));
  }
  amax = block_reduce(amax, OpMax(), smem);
  if (threadIdx.x == 0) row_absmax[row] = amax;
}

// One block folds the n partial maxima: as many waves as four quads a thread need, all requested before the first is
// looked at.  A single wave that asked for 64 quads at a time waited for memory once per 256 maxima.  LayerNorm and
// observer, fp16: 4096 x 1024 10.6 -> 7.0 us, 4096 x 4096 22.8 -> 19.2, 8192 x 8192 59.4 -> 54.4.
constexpr int kLnFinalBlock = 1024;
constexpr int kLnFinalUnroll = 4;
inline unsigned ln_final_threads(int64_t n) {
  const int64_t waves = (n / 4 + kLnFinalUnroll * kWave - 1) / (kLnFinalUnroll * kWave);
  return (unsigned)(waves < 1 ? 1 : (waves < kLnFinalBlock / kWave ? waves : kLnFinalBlock / kWave)) * kWave;
}
__global__ void __launch_bounds__(kLnFinalBlock)
ln_observer_finalize(const float* __restrict__ part, int64_t n, int bits,
                     float* __restrict__ scale, float* __restrict__ zero_point) {
  __shared__ float smem[kLnFinalBlock / kWave];
  const int threads = (int)blockDim.x;
  float amax = 0.0f;
  const int64_t n4 = (reinterpret_cast<uintptr_t>(part) & 15u) == 0 ? n / 4 : 0;
  const f32x4* p4 = reinterpret_cast<const f32x4*>(part);
  for (int64_t i0 = threadIdx.x; i0 < n4; i0 += kLnFinalUnroll * threads) {
    f32x4 q[kLnFinalUnroll];
#pragma unroll
    for (int u = 0; u < kLnFinalUnroll; ++u) {
      const int64_t i = i0 + u * threads;
      q[u] = p4[i < n4 ? i : i0];  // (a maximum twice is the same maximum)
    }
#pragma unroll
    for (int u = 0; u < kLnFinalUnroll; ++u) {
      amax = fmaxf(fmaxf(amax, fmaxf(q[u][0], q[u][1])), fmaxf(q[u][2], q[u][3]));
    }
  }
  for (int64_t i = n4 * 4 + threadIdx.x; i < n; i += threads) amax = fmaxf(amax, part[i]);
  amax = block_reduce(amax, OpMax(), smem);
  if (threadIdx.x == 0) {
    const float denominator = (float)(1 << (bits - 1)) - 1.0f;
    *scale = amax / denominator;
    *zero_point = 0.0f;
  }
}

// ---------------------------------------------------------------------------------------------
// LayerNorm -> observer -> int8 codes without the normalised tensor ever reaching memory
// (ofq_fused_layer_norm_quantization).  fp16 rows of exactly 512 * NP elements with gamma and beta.
// Two kernels:
//   first : the row kernel above without its store: a wave normalises its rows in registers,
//           keeps (mean, inv) of every row and the largest |y| it has seen;
//   second: every block folds the partial maxima into the scale (the arithmetic of
//           ln_observer_finalize, so every block gets the same bits), then a wave reads its rows
//           again -- from L2 where the first kernel left them: the same wave of the same block
//           took them there --, forms y with the stored statistics exactly as the first kernel
//           did, and quantises it the way quantize_half_to_bytes_kernel does.
// Up to 8 rows go to ln_quant_rows below, which needs one launch.
// The codes are those of fused_layer_norm_min_max_observer followed by quantization (symmetric,
// per layer) of its y, bit for bit; traffic is x once from HBM, x once more from L2 and the codes
// (25 MB at 2048 x 4096 where the two ops move 58.7 MB).
// ---------------------------------------------------------------------------------------------
constexpr int kLnqBlock = 512;  // 8 waves: one copy of gamma and beta in LDS serves 8 rows

// gamma and beta of a block: fetched once (wave w fetches pack w of each), parked in LDS, read
// from there pack by pack.  Every wave of the block holding its own copy in registers cost 16 of
// a wave's 24 requests and as much traffic between L2 and the CU as x itself.
template<int NP>
struct LnRowF16 {
  u32x4 graw, braw;
  __device__ __forceinline__ void request(const uint16_t* gamma, const uint16_t* beta, int wave,
                                          int lane) {
    if (wave < NP) {  // the same for every lane of a wave
      graw = *reinterpret_cast<const u32x4*>(gamma + lane * 8 + wave * 512);
      braw = *reinterpret_cast<const u32x4*>(beta + lane * 8 + wave * 512);
    }
  }
  // [gamma NP x 64 pieces][beta NP x 64 pieces]; a barrier must follow before out() is used
  __device__ __forceinline__ void park(u32x4* lds, int wave, int lane) const {
    if (wave < NP) {
      lds[wave * 64 + lane] = graw;
      lds[(NP + wave) * 64 + lane] = braw;
    }
  }
  // y of pack i from the deviations d[8] = x - mean: T(d * inv), * gamma, + beta, each rounded to T
  __device__ __forceinline__ f16x8 out(const float* d, float inv, int i, const u32x4* lds,
                                       int lane) const {
    f16x8 t;
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = (f16)normalised<f16>(d[e], inv);
    t = t * __builtin_bit_cast(f16x8, lds[i * 64 + lane]);
    t = t + __builtin_bit_cast(f16x8, lds[(NP + i) * 64 + lane]);
    return t;
  }
};

// How the codes of one tensor follow from its scale s = absmax / upper: rint(y / s), clamped, NaN -> 0.
//  kLnDivide : the division and the clamp, for any s
//  kLnFast2  : s within 2^+-60: the product with the reciprocal, corrected twice (div_of_half_value)
//  kLnFast1  : 8 bits and the same s: corrected once, which gives the same bits for every |y| <= absmax
//              (quantize_pack.hip, quant_codes8: all fp16 pairs compared; bf16 significands are among them, and
//              a quotient that underflows on the way rounds to 0)
// A fast quotient lies within the codes (y is finite: an infinite one makes the scale infinite), so that
// adding 1.5 * 2^23 leaves the code in the low byte; a NaN that came from a 16-bit value has zeros there.
enum { kLnDivide, kLnFast2, kLnFast1 };
__device__ __forceinline__ int ln_code_mode(float s, int bits) {
  const float mag = __builtin_fabsf(s);
  return !(mag >= 0x1p-60f && mag <= 0x1p60f) ? kLnDivide : bits == 8 ? kLnFast1 : kLnFast2;
}
template<typename T, int MODE>
__device__ __forceinline__ u32x2 ln_codes8(u32x4 y, float s, float recip, int lo, int hi) {
  RawPack<T> r;
  r.q[0] = y;
  float v[8];
  widen<T>(r, v);
  uint32_t words[2];
#pragma unroll
  for (int e4 = 0; e4 < 8; e4 += 4) {
    uint32_t b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a = v[e4 + j];
      if constexpr (MODE == kLnDivide) {
        const float t = __builtin_rintf(a / s);
        int c;
        asm("v_cvt_i32_f32 %0, %1" : "=v"(c) : "v"(t));  // saturates; NaN -> 0
        b[j] = (uint32_t)clamp_i32(c, lo, hi);
      } else {
        float q = a * recip;
        q = __builtin_fmaf(__builtin_fmaf(-s, q, a), recip, q);
        if (MODE == kLnFast2) q = __builtin_fmaf(__builtin_fmaf(-s, q, a), recip, q);
        b[j] = __builtin_bit_cast(uint32_t, q + 12582912.0f);
      }
    }
    words[e4 / 4] = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u)
                    | __builtin_amdgcn_perm(b[3], b[2], 0x04000c0cu);
  }
  return u32x2{words[0], words[1]};
}

// f(constant) for the mode of this scale, taken once per wave: inside a loop every quotient would be computed
// and one selected
template<typename F>
__device__ __forceinline__ void ln_with_mode(float s, int bits, F&& f) {
  const int mode = ln_code_mode(s, bits);
  if (mode == kLnFast1) f(std::integral_constant<int, kLnFast1>());
  else if (mode == kLnFast2) f(std::integral_constant<int, kLnFast2>());
  else f(std::integral_constant<int, kLnDivide>());
}

template<int NP, bool EXACT>
__global__ void __launch_bounds__(kLnqBlock)
ln_quant_first(const uint16_t* __restrict__ x, const uint16_t* __restrict__ gamma,
               const uint16_t* __restrict__ beta, float* __restrict__ block_absmax,
               float* __restrict__ stats, int64_t rows, double eps64) {
  constexpr int kCols = NP * 512;
  constexpr int kWaves = kLnqBlock / kWave;
  __shared__ float wmax[kWaves];
  __shared__ u32x4 params[2 * NP * 64];
  const float eps = (float)eps64;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t gw = (int64_t)blockIdx.x * kWaves + wave;
  const int64_t nwaves = (int64_t)gridDim.x * kWaves;
  LnRowF16<NP> prm;
  prm.request(gamma, beta, wave, lane);
  u32x4 cur[NP];
  {
    // (a wave past the last row re-reads row 0 and skips the loop: it only joins the barriers)
    const uint16_t* xr = x + (gw < rows ? gw : 0) * kCols + lane * 8;
#pragma unroll
    for (int i = 0; i < NP; ++i) cur[i] = *reinterpret_cast<const u32x4*>(xr + i * 512);
  }
  prm.park(params, wave, lane);
  __syncthreads();
  f16x8 amax8 = {(f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f};
  for (int64_t row = gw; row < rows; row += nwaves) {
    if (row != gw) {
      const uint16_t* xr = x + row * kCols + lane * 8;
#pragma unroll
      for (int i = 0; i < NP; ++i) cur[i] = *reinterpret_cast<const u32x4*>(xr + i * 512);
    }
    float f[NP][8];
    float sum = 0.0f;
    double sum64 = 0.0;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      RawPack<f16> rp;
      rp.q[0] = cur[i];
      widen<f16>(rp, f[i]);
      if constexpr (EXACT) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sum64 += (double)f[i][e];
      } else {
        uint32_t ones_bits = 0x3c003c00u;  // (1, 1) held in a register, see ln_observer_wave_full
        asm volatile("" : "+v"(ones_bits));
        const f16x2 ones = __builtin_bit_cast(f16x2, ones_bits);
        const f16x8 h = __builtin_bit_cast(f16x8, cur[i]);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 0, 1), ones, sum, false);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 2, 3), ones, sum, false);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 4, 5), ones, sum, false);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 6, 7), ones, sum, false);
      }
    }
    float mean, inv;
    if constexpr (EXACT) {
      sum64 = wave_reduce(sum64, OpSum());
      const double mean64 = sum64 / (double)kCols;
      mean = (float)mean64;
      double q = 0.0;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const double d = (double)f[i][e] - mean64;
          q = __builtin_fma(d, d, q);
          f[i][e] = f[i][e] - mean;
        }
      }
      q = wave_reduce(q, OpSum());
      inv = exact_inv(q, (double)kCols, eps64);
    } else {
      sum = wave_reduce(sum, OpSum());
      mean = sum / (float)kCols;
      float m2 = 0.0f;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          f[i][e] = f[i][e] - mean;
          m2 = __builtin_fmaf(f[i][e], f[i][e], m2);
        }
      }
      m2 = wave_reduce(m2, OpSum());
      const float var = fmaxf(m2 / (float)kCols, 0.0f);
      inv = 1.0f / __builtin_sqrtf(var + eps);
    }
    if (lane == 0) {
      stats[2 * row] = mean;
      stats[2 * row + 1] = inv;
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const u32x4 tb = __builtin_bit_cast(u32x4, prm.out(f[i], inv, i, params, lane));
      const u32x4 ab = {tb[0] & 0x7FFF7FFFu, tb[1] & 0x7FFF7FFFu, tb[2] & 0x7FFF7FFFu,
                        tb[3] & 0x7FFF7FFFu};
      amax8 = __builtin_elementwise_max(amax8, __builtin_bit_cast(f16x8, ab));
    }
  }
  float amax = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) amax = fmaxf(amax, (float)amax8[e]);
  amax = wave_reduce(amax, OpMax());
  // one partial maximum per block, so that the second kernel folds them with one request
  if (lane == 0) wmax[wave] = amax;
  __syncthreads();
  if (threadIdx.x == 0) {
    amax = wmax[0];
#pragma unroll
    for (int wv = 1; wv < kWaves; ++wv) amax = fmaxf(amax, wmax[wv]);
    block_absmax[blockIdx.x] = amax;
  }
}

// SPLIT: a row is taken by SPLIT waves of SPLIT different blocks, NP / SPLIT packs each (nothing
// in this kernel crosses the lanes of a row), so that few rows still make enough waves to
// overlap one wave's arithmetic with another's requests.  Block b works on the rows of block
// p = (b / (8 * SPLIT)) * 8 + b % 8 of the first kernel, part (b / 8) % SPLIT: b and p agree
// modulo 8, the number of XCDs the blocks are dealt over, so a row is read again through the L2
// that holds it.  The grid is ceil(first_grid / 8) * 8 * SPLIT blocks.
template<int NP, int SPLIT>
__global__ void __launch_bounds__(kLnqBlock)
ln_quant_second(const uint16_t* __restrict__ x, const uint16_t* __restrict__ gamma,
                const uint16_t* __restrict__ beta, const float* __restrict__ part, int64_t nparts,
                const float* __restrict__ stats, int8_t* __restrict__ codes,
                float* __restrict__ scale, float* __restrict__ zero_point, int64_t rows, int bits,
                int first_grid) {
  static_assert(NP % SPLIT == 0, "whole packs per part");
  constexpr int kCols = NP * 512;
  constexpr int NPW = NP / SPLIT;  // packs of a row this wave takes
  constexpr int kWaves = kLnqBlock / kWave;
  __shared__ float wmax[kWaves];
  __shared__ u32x4 params[2 * NPW * 64];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t fb = ((int64_t)blockIdx.x / (8 * SPLIT)) * 8 + blockIdx.x % 8;
  const int part_of_row = (int)((blockIdx.x / 8) % SPLIT);
  const int pack0 = part_of_row * NPW;
  const int64_t gw = fb * kWaves + wave;
  const int64_t nwaves = (int64_t)first_grid * kWaves;
  const bool active = gw < rows;
  // Requests in the order of their use: the partial maxima (one 16-byte piece per thread:
  // nparts <= 512 <= 4 * kLnqBlock), the statistics of the wave's first row, the wave's share of
  // the parameters, then the row, so that the maxima can be folded and the parameters parked
  // while the row is still on its way.
  const int64_t n4 = (nparts + 3) / 4;
  const int64_t pidx = (int64_t)threadIdx.x < n4 ? threadIdx.x : 0;
  f32x4 pq = reinterpret_cast<const f32x4*>(part)[pidx];
  const float* st0 = stats + 2 * (active ? gw : 0);
  float mean0 = st0[0], inv0 = st0[1];
  LnRowF16<NPW> prm;
  prm.request(gamma + pack0 * 512, beta + pack0 * 512, wave, lane);
  u32x4 cur[NPW];
  {
    const uint16_t* xr = x + (active ? gw : 0) * kCols + pack0 * 512 + lane * 8;
#pragma unroll
    for (int i = 0; i < NPW; ++i) cur[i] = *reinterpret_cast<const u32x4*>(xr + i * 512);
  }
  prm.park(params, wave, lane);
  // scale = max of the partial maxima / (2^(bits-1) - 1), the same operations in every block
  // (the last piece may reach up to three floats past the partials: masked)
  float amax = 0.0f;
  {
#pragma unroll
    for (int e = 0; e < 4; ++e) amax = fmaxf(amax, pidx * 4 + e < nparts ? pq[e] : 0.0f);
    amax = wave_reduce(amax, OpMax());
    if (lane == 0) wmax[wave] = amax;
    __syncthreads();  // (also orders the parked parameters before their use)
    amax = 0.0f;
#pragma unroll
    for (int wv = 0; wv < kWaves; ++wv) amax = fmaxf(amax, wmax[wv]);
  }
  const float upper = (float)(1 << (bits - 1)) - 1.0f;
  const float s = amax / upper;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *scale = s;
    *zero_point = 0.0f;
  }
  if (!active) return;
  const float recip = 1.0f / s;
  const int hi = (int)upper, lo = -hi - 1;
  ln_with_mode(s, bits, [&](auto mode) {
    for (int64_t row = gw; row < rows; row += nwaves) {
      if (row != gw) {
        const uint16_t* xr = x + row * kCols + pack0 * 512 + lane * 8;
#pragma unroll
        for (int i = 0; i < NPW; ++i) cur[i] = *reinterpret_cast<const u32x4*>(xr + i * 512);
      }
      float mean = mean0, inv = inv0;
      if (row != gw) {
        mean = stats[2 * row];
        inv = stats[2 * row + 1];
      }
      int8_t* cr = codes + row * kCols + pack0 * 512 + lane * 8;
#pragma unroll
      for (int i = 0; i < NPW; ++i) {
        RawPack<f16> rp;
        rp.q[0] = cur[i];
        float d[8];
        widen<f16>(rp, d);
#pragma unroll
        for (int e = 0; e < 8; ++e) d[e] = d[e] - mean;
        // (held as four packed registers: otherwise the affine is emitted element by element)
        u32x4 yb = __builtin_bit_cast(u32x4, prm.out(d, inv, i, params, lane));
        asm volatile("" : "+v"(yb[0]), "+v"(yb[1]), "+v"(yb[2]), "+v"(yb[3]));
        const u32x2 w2 = ln_codes8<f16, decltype(mode)::value>(yb, s, recip, lo, hi);
        __builtin_nontemporal_store(w2, reinterpret_cast<u32x2*>(cr + i * 512));
      }
    }
  });
}

// ---------------------------------------------------------------------------------------------
// The same composition for fp16 and bf16 rows of any 8 * n elements up to 16384, gamma and beta each
// optional.  A row is taken by WPR waves: one (the arithmetic of ln_observer_wave_rows; FULL:
// rows of 512 * NP elements, fp16 with the row sum of ln_observer_wave_full) or four (that of ln_observer_rows), so scale and codes carry
// the bits of the two ops.
//   ln_quant_rows<kLnStats> + ln_quant_codes : two launches; y is formed twice and never stored
//   ln_quant_rows<kLnCodes>                  : one launch of one block, for as many rows as it holds
//     (8, or 4 of more than 4096 elements): the rows wait in registers for the block's maximum
// Time of a call of the two ops and of this: 1 x 2432 fp16 13.0 -> 6.4 us, 8 x 1280 bf16 13.6 -> 6.4, 64 x 6080
// fp16 13.3 -> 9.2, 1024 x 6080 19.1 -> 14.0, 4096 x 4096 bf16 44 -> 31 (host-bound up to some hundred rows:
// three launches and two allocations became one or two launches).  Many rows are bound by the vector units
// of both kernels: 8192 x 2432 fp16 17.8 + 15.3 us, where their traffic takes about 14.
// ln_quant_rows<OUT = kLnY> is also the observer of few rows, with or without a residual input.
// ---------------------------------------------------------------------------------------------
constexpr int ln_rows_per_block(int wpr, bool one) { return wpr == 1 ? 8 : one ? 4 : 1; }

template<typename T>
__device__ __forceinline__ RawPack<T> load_pack(const uint16_t* p) {
  return load_raw<T>(reinterpret_cast<const typename TT<T>::storage*>(p));
}

// 8 floats rounded to bf16, two to an instruction; the packed values, and optionally the floats again
__device__ __forceinline__ u32x4 round8_bf16(float* f, bool again) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{f[2 * i], f[2 * i + 1]}, bf2));
    asm volatile("" : "+v"(w));  // (or the pair is converted one by one where it is widened again)
    r[i] = w;
    if (again) {
      f[2 * i] = __builtin_bit_cast(float, w << 16);
      f[2 * i + 1] = __builtin_bit_cast(float, w & 0xFFFF0000u);
    }
  }
  return r;
}

// What stands for an absent parameter or residual input, so that nothing is decided per element: gamma 1; beta +0
// next to a gamma (the reference adds its default beta 0: -0 becomes +0) and else -0, which leaves every value as
// it is; +0 for a residual input
template<typename T>
__device__ __forceinline__ uint32_t ln_ones() {
  return TT<T>::dtype == OFQ_F16 ? 0x3C003C00u : 0x3F803F80u;
}
template<typename T>
__device__ __forceinline__ RawPack<T> ln_pack_or(const uint16_t* p, int64_t at, uint32_t absent) {
  RawPack<T> r;
  r.q[0] = u32x4{absent, absent, absent, absent};
  if (p) r = load_pack<T>(p + at);
  return r;
}

// y of 8 elements from their deviations x - mean, as ln_observer_wave_rows forms it
template<typename T>
__device__ __forceinline__ u32x4 ln_out8(const float* d, float inv, const RawPack<T>& g, const RawPack<T>& b) {
  if constexpr (TT<T>::dtype == OFQ_F16) {
    f16x8 t;
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = (f16)normalised<f16>(d[e], inv);
    t = t * __builtin_bit_cast(f16x8, g.q[0]);
    t = t + __builtin_bit_cast(f16x8, b.q[0]);
    u32x4 bits = __builtin_bit_cast(u32x4, t);
    // (held as four packed registers: otherwise the affine is emitted element by element)
    asm volatile("" : "+v"(bits[0]), "+v"(bits[1]), "+v"(bits[2]), "+v"(bits[3]));
    return bits;
  } else {
    float gf[8], bf[8], t[8];
    widen<T>(g, gf);
    widen<T>(b, bf);
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = d[e] * inv;
    round8_bf16(t, true);
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = t[e] * gf[e];
    round8_bf16(t, true);
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = t[e] + bf[e];
    return round8_bf16(t, false);
  }
}

// the largest |y| seen, NaN passed over: fp16 in eight packed maxima, bf16 in one float
template<typename T>
struct LnAbsMax {
  f16x8 packed = {(f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f, (f16)0.0f};
  float one = 0.0f;
  __device__ __forceinline__ void take(u32x4 y) {
    if constexpr (TT<T>::dtype == OFQ_F16) {
      const u32x4 ab = {y[0] & 0x7FFF7FFFu, y[1] & 0x7FFF7FFFu, y[2] & 0x7FFF7FFFu, y[3] & 0x7FFF7FFFu};
      packed = __builtin_elementwise_max(packed, __builtin_bit_cast(f16x8, ab));
    } else {
      RawPack<T> r;
      r.q[0] = y;
      float v[8];
      widen<T>(r, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) one = fmaxf(one, fabsf(v[e]));
    }
  }
  __device__ __forceinline__ float value() const {
    float m = one;
#pragma unroll
    for (int e = 0; e < 8; ++e) m = fmaxf(m, (float)packed[e]);
    return m;
  }
};

// the sum over the WPR waves of a row, in the order of block_reduce (every thread of the block calls it)
template<int WPR, typename V>
__device__ __forceinline__ V row_sum(V v, V* smem) {
  v = wave_reduce(v, OpSum());
  if constexpr (WPR == 1) return v;
  const int wave = threadIdx.x / kWave;
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0) smem[wave] = v;
  __syncthreads();
  const int w0 = wave / WPR * WPR;
  V r = smem[w0];
#pragma unroll
  for (int i = 1; i < WPR; ++i) r = r + smem[w0 + i];
  return r;
}

// the residual inputs of skip_layer_norm, see SkipArgs
struct LnSkip16 {
  const uint16_t *bias, *skip;
  float alpha;
};

// 8 elements of the residual sum in place of those of x: b bias, s skip
template<typename T>
__device__ __forceinline__ void ln_add_skip(RawPack<T>& v, float alpha, const RawPack<T>& s,
                                            const RawPack<T>& b) {
  if constexpr (TT<T>::dtype == OFQ_F16) {  // (native fp16 arithmetic, see ln_observer_wave_full)
    const f16x8 xb = __builtin_bit_cast(f16x8, v.q[0]) + __builtin_bit_cast(f16x8, b.q[0]);
    v.q[0] = __builtin_bit_cast(u32x4, xb + __builtin_bit_cast(f16x8, s.q[0]) * (f16)alpha);
  } else {
    float fx[8], fb[8], fs[8];
    widen<T>(v, fx);
    widen<T>(b, fb);
    widen<T>(s, fs);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      fx[e] = fx[e] + fb[e];
      fs[e] = fs[e] * alpha;
    }
    round8_bf16(fx, true);
    round8_bf16(fs, true);
#pragma unroll
    for (int e = 0; e < 8; ++e) fx[e] = fx[e] + fs[e];
    v.q[0] = round8_bf16(fx, false);
  }
}

// What a launch leaves: (mean, inv) of the rows and a maximum per block, or, of one block, codes or y
enum { kLnStats, kLnCodes, kLnY };

template<typename T, int NP, int WPR, bool FULL, bool EXACT, int OUT, bool SKIP>
__global__ void __launch_bounds__(ln_rows_per_block(WPR, OUT != kLnStats) * WPR * kWave)
ln_quant_rows(const uint16_t* __restrict__ x, const uint16_t* __restrict__ gamma,
              const uint16_t* __restrict__ beta, float* __restrict__ block_absmax,
              float* __restrict__ stats, void* __restrict__ out, float* __restrict__ scale,
              float* __restrict__ zero_point, int64_t rows, int cols, double eps64, int bits, LnSkip16 sk) {
  constexpr bool ONE = OUT != kLnStats;
  static_assert(ONE || !SKIP, "the residual variant has one block");
  constexpr int kRows = ln_rows_per_block(WPR, ONE);
  constexpr int kWaves = kRows * WPR;
  constexpr int kStep = WPR * kWave;  // packs between two of a thread
  __shared__ float smem[kWaves];
  __shared__ double smem64[EXACT ? kWaves : 1];
  const float eps = (float)eps64;
  const int t = threadIdx.x % kStep;
  const int npacks = cols / 8;
  const int per_block = ONE ? kRows : (int)blockDim.x / kStep;
  const int64_t first = (int64_t)blockIdx.x * per_block + threadIdx.x / kStep;
  const int64_t stride = (int64_t)gridDim.x * per_block;
  // rows of a block in turns that all its threads take (row_sum holds barriers); a thread whose row lies past
  // the last one reads nothing
  const int64_t turns = ONE ? 1 : (rows - (int64_t)blockIdx.x * per_block + stride - 1) / stride;
  // gamma and beta: one copy in LDS for the rows of a block, or in the registers of the only row's threads
  constexpr bool kShared = kRows > 1;
  __shared__ u32x4 params[kShared ? 2 * NP * kStep : 1];
  const uint32_t no_beta = gamma ? 0u : 0x80008000u;
  RawPack<T> gr[kShared ? 1 : NP], br[kShared ? 1 : NP], v[NP];
  bool in[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    in[i] = FULL || t + i * kStep < npacks;
    if constexpr (!kShared) {
      if (in[i]) {
        gr[i] = ln_pack_or<T>(gamma, (t + i * kStep) * 8, ln_ones<T>());
        br[i] = ln_pack_or<T>(beta, (t + i * kStep) * 8, no_beta);
      }
    }
  }
  auto request = [&](int64_t row) {
    const uint16_t* xr = x + (row < rows ? row : 0) * cols;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if (in[i] && row < rows) v[i] = load_pack<T>(xr + (t + i * kStep) * 8);
      else v[i].q[0] = u32x4{0u, 0u, 0u, 0u};
    }
  };
  request(first);
  RawPack<T> sr[SKIP ? NP : 1], br1[SKIP ? NP : 1];
  if constexpr (SKIP) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if (in[i] && first < rows) {
        sr[i] = ln_pack_or<T>(sk.skip, first * cols + (t + i * kStep) * 8, 0u);
        br1[i] = ln_pack_or<T>(sk.bias, (t + i * kStep) * 8, 0u);
      }
    }
  }
  if constexpr (kShared) {
    // all requested before the first is stored: a block of one wave, which takes NP packs of each, waited for
    // memory NP times (10 x 4096 bf16 to codes 10.2 -> 9.0 us, 15 x 3784 fp16 10.2 -> 9.0)
    constexpr int kTurns = ONE ? (NP + kRows - 1) / kRows : NP;
    RawPack<T> g[kTurns], b[kTurns];
#pragma unroll
    for (int i = 0; i < kTurns; ++i) {
      const int p = threadIdx.x + i * blockDim.x;
      if (p < npacks) {
        g[i] = ln_pack_or<T>(gamma, p * 8, ln_ones<T>());
        b[i] = ln_pack_or<T>(beta, p * 8, no_beta);
      }
    }
#pragma unroll
    for (int i = 0; i < kTurns; ++i) {
      const int p = threadIdx.x + i * blockDim.x;
      if (p < npacks) {
        params[p] = g[i].q[0];
        params[NP * kStep + p] = b[i].q[0];
      }
    }
    __syncthreads();
  }
  // The rows of many blocks are held in storage format and widened again in every pass: without the empty asm
  // the compiler keeps the widened floats too, twice the registers (176 to 240 of them for rows of 4096).
  auto hold_pack = [](RawPack<T>& r) {
    u32x4 h = r.q[0];
    asm volatile("" : "+v"(h[0]), "+v"(h[1]), "+v"(h[2]), "+v"(h[3]));
    r.q[0] = h;
  };
  auto hold = [&]() {
    if constexpr (ONE && !(EXACT && WPR > 1)) return;
#pragma unroll
    for (int i = 0; i < NP; ++i) hold_pack(v[i]);
  };
  LnAbsMax<T> amax8;
  float mean = 0.0f, inv = 0.0f;
  for (int64_t turn = 0; turn < turns; ++turn) {
    const int64_t row = first + turn * stride;
    const bool live = row < rows;
    if (turn != 0) request(row);
    if constexpr (SKIP) {
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        if (in[i] && live) ln_add_skip<T>(v[i], sk.alpha, sr[i], br1[i]);
      }
    }
    // (an element past the row adds a zero to the sum and, skipped, nothing to the squares)
    float sum = 0.0f;
    double sum64 = 0.0;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      float f[8];
      widen<T>(v[i], f);
      if constexpr (EXACT) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sum64 += (double)f[e];
      } else if constexpr (FULL && TT<T>::dtype == OFQ_F16) {
        uint32_t ones_bits = 0x3c003c00u;  // (1, 1) held in a register, see ln_observer_wave_full
        asm volatile("" : "+v"(ones_bits));
        const f16x2 ones = __builtin_bit_cast(f16x2, ones_bits);
        const f16x8 h = __builtin_bit_cast(f16x8, v[i].q[0]);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 0, 1), ones, sum, false);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 2, 3), ones, sum, false);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 4, 5), ones, sum, false);
        sum = __builtin_amdgcn_fdot2(__builtin_shufflevector(h, h, 6, 7), ones, sum, false);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) sum += f[e];
      }
    }
    if constexpr (EXACT) {
      sum64 = row_sum<WPR>(sum64, smem64);
      hold();
      const double mean64 = sum64 / (double)cols;
      double q = 0.0;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        if (!in[i]) continue;
        float f[8];
        widen<T>(v[i], f);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const double d = (double)f[e] - mean64;
          q = __builtin_fma(d, d, q);
        }
      }
      q = row_sum<WPR>(q, smem64);
      mean = (float)mean64;
      inv = exact_inv(q, (double)cols, eps64);
    } else {
      sum = row_sum<WPR>(sum, smem);
      hold();
      mean = sum / (float)cols;
      float m2 = 0.0f;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        if (!in[i]) continue;
        float f[8];
        widen<T>(v[i], f);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = f[e] - mean;
          m2 = __builtin_fmaf(d, d, m2);
        }
      }
      m2 = row_sum<WPR>(m2, smem);
      const float var = fmaxf(m2 / (float)cols, 0.0f);
      inv = 1.0f / __builtin_sqrtf(var + eps);
    }
    hold();
    if constexpr (!ONE) {
      if (t == 0 && live) {
        stats[2 * row] = mean;
        stats[2 * row + 1] = inv;
      }
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if (!in[i] || !live) continue;
      float d[8];
      widen<T>(v[i], d);
#pragma unroll
      for (int e = 0; e < 8; ++e) d[e] = d[e] - mean;
      RawPack<T> g, b;
      if constexpr (kShared) {
        g.q[0] = params[t + i * kStep];
        b.q[0] = params[NP * kStep + t + i * kStep];
      } else {
        hold_pack(gr[i]), hold_pack(br[i]);  // (or their floats are kept over the turns)
        g = gr[i], b = br[i];
      }
      const u32x4 y = ln_out8<T>(d, inv, g, b);
      amax8.take(y);
      if constexpr (OUT == kLnCodes) v[i].q[0] = y;
      if constexpr (OUT == kLnY) {
        *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(out) + row * cols + (t + i * kStep) * 8) = y;
      }
    }
  }
  const float amax = block_reduce(amax8.value(), OpMax(), smem);
  if constexpr (!ONE) {
    if (threadIdx.x == 0) block_absmax[blockIdx.x] = amax;
  } else {
    const float upper = (float)(1 << (bits - 1)) - 1.0f;
    const float s = amax / upper;
    if (threadIdx.x == 0) {
      *scale = s;
      *zero_point = 0.0f;
    }
    if (OUT != kLnCodes || first >= rows) return;
    int8_t* codes = static_cast<int8_t*>(out);
    const float recip = 1.0f / s;
    const int hi = (int)upper, lo = -hi - 1;
    ln_with_mode(s, bits, [&](auto mode) {
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        if (!in[i]) continue;
        *reinterpret_cast<u32x2*>(codes + first * cols + (t + i * kStep) * 8) =
            ln_codes8<T, decltype(mode)::value>(v[i].q[0], s, recip, lo, hi);
      }
    });
  }
}

// Codes from the statistics of ln_quant_rows.  A thread keeps one pack of gamma and of beta and walks the rows
// blockIdx.y, + gridDim.y, ..., U of them requested at once; every block folds the partial maxima into the
// scale by itself.
constexpr int kLnCodesBlock = 256;
template<typename T, int U>
__global__ void __launch_bounds__(kLnCodesBlock)
ln_quant_codes(const uint16_t* __restrict__ x, const uint16_t* __restrict__ gamma,
               const uint16_t* __restrict__ beta, const float* __restrict__ part, int nparts,
               const float* __restrict__ stats, int8_t* __restrict__ codes, float* __restrict__ scale,
               float* __restrict__ zero_point, int64_t rows, int cols, int bits) {
  __shared__ float smem[kLnCodesBlock / kWave];
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  const bool in = p < cols / 8;
  const int at = in ? p * 8 : 0;
  RawPack<T> v[U], g, b;
  float mean[U], inv[U];
  auto request = [&](int64_t row0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t row = row0 + u * (int64_t)gridDim.y;
      const int64_t r = row < rows ? row : blockIdx.y;
      v[u] = load_pack<T>(x + r * cols + at);
      mean[u] = stats[2 * r];
      inv[u] = stats[2 * r + 1];
    }
  };
  float amax = 0.0f;
  for (int i = threadIdx.x; i < nparts; i += blockDim.x) amax = fmaxf(amax, part[i]);
  request(blockIdx.y);
  g = ln_pack_or<T>(gamma, at, ln_ones<T>());
  b = ln_pack_or<T>(beta, at, gamma ? 0u : 0x80008000u);
  amax = block_reduce(amax, OpMax(), smem);
  const float upper = (float)(1 << (bits - 1)) - 1.0f;
  const float s = amax / upper;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
    *scale = s;
    *zero_point = 0.0f;
  }
  if (!in) return;
  const float recip = 1.0f / s;
  const int hi = (int)upper, lo = -hi - 1;
  ln_with_mode(s, bits, [&](auto mode) {
    for (int64_t row0 = blockIdx.y; row0 < rows; row0 += U * (int64_t)gridDim.y) {
      if (row0 != blockIdx.y) request(row0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t row = row0 + u * (int64_t)gridDim.y;
        if (row >= rows) break;
        float d[8];
        widen<T>(v[u], d);
#pragma unroll
        for (int e = 0; e < 8; ++e) d[e] = d[e] - mean[u];
        const u32x4 y = ln_out8<T>(d, inv[u], g, b);
        *reinterpret_cast<u32x2*>(codes + row * cols + at) =
            ln_codes8<T, decltype(mode)::value>(y, s, recip, lo, hi);
      }
    }
  });
}

// host-side rounding of a float to T (round to nearest even)
template<typename T>
float round_to_T_host(float v) {
  if (TT<T>::dtype == OFQ_F16) return (float)(_Float16)v;
  if (TT<T>::dtype == OFQ_BF16) {
    uint32_t u;
    __builtin_memcpy(&u, &v, 4);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return v;  // NaN stays NaN
    u += 0x7FFFu + ((u >> 16) & 1u);
    u &= 0xFFFF0000u;
    __builtin_memcpy(&v, &u, 4);
    return v;
  }
  return v;
}

struct LnQuantArgs {
  const uint16_t *x, *gamma, *beta;
  float *part, *stats;
  void* out;
  float *scale, *zero_point;
  int64_t rows;
  int cols;
  double eps;
  int bits;
};

// Rows that one block takes; 0 for rows longer than it takes.  One launch of 4 x 4096, 8 x 4096 and 4 x 8192 fp16
// rows with a residual input is 5.0, 6.6 and 7.1 us, the row kernel and the fold 4.1 + 1.4, 4.6 + 1.4 and
// 7.3 + 1.5 with a gap between them and 2.3 us of the host for the second launch.  For y of long bf16 rows, which
// take more of the one CU's vector units, it ends earlier: 4 x 4096 6.6, 8 x 4096 8.9 and 4 x 8192 9.8 us
// against 6.4 + 1.2, 7.1 + 1.4 and 7.7 + 1.2.
template<typename T>
constexpr int ln_one_block_rows(int packs, int out) {
  const int rows = packs <= 8 * kWave ? ln_rows_per_block(1, true)
                   : packs <= 16 * kWave ? ln_rows_per_block(4, true) : 0;
  return TT<T>::dtype == OFQ_BF16 && out == kLnY && packs > 4 * kWave ? rows / 2 : rows;
}

template<typename T, int NP, int WPR, bool FULL, bool EXACT, int OUT, bool SKIP>
void launch_ln_one_block(hipStream_t st, const LnQuantArgs& a, const LnSkip16& sk) {
  ln_quant_rows<T, NP, WPR, FULL, EXACT, OUT, SKIP><<<1, ln_rows_per_block(WPR, true) * WPR * kWave, 0, st>>>(
      a.x, a.gamma, a.beta, a.part, a.stats, a.out, a.scale, a.zero_point, a.rows, a.cols, a.eps, a.bits, sk);
}

// fp16 rows are full only with both parameters, as for ln_observer_wave_full, whose sums those are
template<typename T, bool EXACT, int OUT, bool SKIP>
void ln_one_block(hipStream_t st, const LnQuantArgs& a, const LnSkip16& sk) {
  const int packs = a.cols / 8;
  const bool full = (a.cols == 512 || a.cols == 1024 || a.cols == 2048 || a.cols == 4096)
                    && (TT<T>::dtype != OFQ_F16 || (a.gamma != nullptr && a.beta != nullptr));
#define OFQ_LN_ONE(NPV)                                                                \
  if (full) launch_ln_one_block<T, NPV, 1, true, EXACT, OUT, SKIP>(st, a, sk);         \
  else launch_ln_one_block<T, NPV, 1, false, EXACT, OUT, SKIP>(st, a, sk)
  if (packs <= kWave) {
    OFQ_LN_ONE(1);
  } else if (packs <= 2 * kWave) {
    OFQ_LN_ONE(2);
  } else if (packs <= 4 * kWave) {
    OFQ_LN_ONE(4);
  } else if (packs <= 8 * kWave) {
    OFQ_LN_ONE(8);
  } else {
    launch_ln_one_block<T, 4, 4, false, EXACT, OUT, SKIP>(st, a, sk);
  }
#undef OFQ_LN_ONE
}

template<typename T, int NP, int WPR, bool EXACT>
void launch_ln_quant_rows(hipStream_t st, const LnQuantArgs& a) {
  constexpr int kMany = ln_rows_per_block(WPR, false);
  // a row to a block until every CU has one, to a SIMD until those have one, then 16 waves per CU
  int8_t* codes = static_cast<int8_t*>(a.out);
  const int per_block = a.rows <= 256 ? 1 : a.rows <= 1024 && kMany > 4 ? 4 : kMany;
  const int64_t blocks = (a.rows + per_block - 1) / per_block, most = 4096 / (kMany * WPR);
  const int grid = (int)(blocks < most ? blocks : most);
  ln_quant_rows<T, NP, WPR, false, EXACT, kLnStats, false><<<grid, per_block * WPR * kWave, 0, st>>>(
      a.x, a.gamma, a.beta, a.part, a.stats, codes, a.scale, a.zero_point, a.rows, a.cols, a.eps, a.bits, LnSkip16{});
  const int packs = a.cols / 8;
  const int bx = (packs + kLnCodesBlock - 1) / kLnCodesBlock;
  const int threads = ((packs + bx - 1) / bx + kWave - 1) / kWave * kWave;
  const int most_y = 8192 / (bx * threads / kWave);
  if (a.rows <= most_y) {
    ln_quant_codes<T, 1><<<dim3(bx, (unsigned)a.rows), threads, 0, st>>>(
        a.x, a.gamma, a.beta, a.part, grid, a.stats, codes, a.scale, a.zero_point, a.rows, a.cols, a.bits);
  } else {
    const int64_t turns = (a.rows + 4 * (int64_t)most_y - 1) / (4 * (int64_t)most_y);
    const unsigned by = (unsigned)((a.rows + 4 * turns - 1) / (4 * turns));
    ln_quant_codes<T, 4><<<dim3(bx, by), threads, 0, st>>>(
        a.x, a.gamma, a.beta, a.part, grid, a.stats, codes, a.scale, a.zero_point, a.rows, a.cols, a.bits);
  }
}

template<typename T, bool SKIP, bool EXACT>
int launch(hipStream_t st, const void* x, const void* gamma, const void* beta, void* y,
           float* scale, float* zero_point, int64_t rows, int64_t cols, double eps, int bits,
           float* ws, const void* bias, const void* skip, double alpha) {
  typedef typename TT<T>::storage S;
  const S* xs = static_cast<const S*>(x);
  const S* gs = static_cast<const S*>(gamma);
  const S* bs = static_cast<const S*>(beta);
  S* ys = static_cast<S*>(y);
  SkipArgs<T> sk;
  sk.bias = static_cast<const S*>(bias);
  sk.skip = static_cast<const S*>(skip);
  // T(alpha): the reference casts its float alpha to T (skip_layer_norm_kernel.cu:36,62)
  sk.alpha = round_to_T_host<T>((float)alpha);
  const bool vec_ok = cols % 8 == 0 && ofq_aligned16(x) && ofq_aligned16(y)
                      && ofq_aligned16(gamma) && ofq_aligned16(beta) && ofq_aligned16(bias)
                      && ofq_aligned16(skip) && (cols * sizeof(S)) % 16 == 0;
  const int64_t npacks = cols / 8;
  if constexpr (sizeof(S) == 2) {
    // as many rows as one block holds need no second launch
    if (vec_ok && npacks <= 16 * kWave && rows <= ln_one_block_rows<T>((int)npacks, kLnY)) {
      const auto u16 = [](const void* p) { return static_cast<const uint16_t*>(p); };
      const LnQuantArgs a = {u16(x), u16(gamma), u16(beta), nullptr, nullptr, y, scale, zero_point, rows,
                             (int)cols, eps, bits};
      ln_one_block<T, EXACT, kLnY, SKIP>(st, a, LnSkip16{u16(bias), u16(skip), sk.alpha});
      return ofq_check_launch();
    }
  }
  int64_t nparts = rows;
  constexpr int kWavesPerBlock = kLnBlock / kWave;
  // fp32 rows beyond 2048 elements would not fit a lane's registers at two waves per SIMD
  const int64_t wave_packs = (sizeof(S) == 4 ? 4 : 8) * kWave;
  if constexpr (sizeof(S) == 2) {
    const int np = (int)(cols / 512);
    if (vec_ok && gamma != nullptr && beta != nullptr && cols % 512 == 0
        && (np == 1 || np == 2 || np == 4 || np == 8)) {
      // one row per wave while the rows fit 16 waves per CU; beyond that 8 waves per CU walk the
      // rows with the next row in flight
      const bool loop = rows > 256 * 16;
      // (the residual variant at NP = 8 holds 230 registers: 8 waves per CU there as well)
      const int64_t waves = loop ? 256 * 8 : rows;
      const int grid = (int)((waves + kWavesPerBlock - 1) / kWavesPerBlock);
      nparts = waves;
#define OFQ_LN_FULL(NPV)                                                                        \
  if (SKIP) {                                                                                    \
    ln_observer_wave_full<T, NPV, false, SKIP, EXACT><<<grid, kLnBlock, 0, st>>>(                \
        xs, gs, bs, ys, ws, rows, eps, sk);                                                      \
  } else if (loop) {                                                                             \
    ln_observer_wave_full<T, NPV, true, false, EXACT><<<grid, kLnBlock, 0, st>>>(                \
        xs, gs, bs, ys, ws, rows, eps, sk);                                                      \
  } else {                                                                                       \
    ln_observer_wave_full<T, NPV, false, false, EXACT><<<grid, kLnBlock, 0, st>>>(               \
        xs, gs, bs, ys, ws, rows, eps, sk);                                                      \
  }
      switch (np) {
        case 1: OFQ_LN_FULL(1) break;
        case 2: OFQ_LN_FULL(2) break;
        case 4: OFQ_LN_FULL(4) break;
        default: OFQ_LN_FULL(8) break;
      }
#undef OFQ_LN_FULL
      ln_observer_finalize<<<1, ln_final_threads(nparts), 0, st>>>(ws, nparts, bits, scale, zero_point);
      return ofq_check_launch();
    }
  }
  if (vec_ok && npacks <= wave_packs) {
    // about 32 KB of rows in flight per CU streams best: 4 waves per CU for 8 KB rows, up to 16
    // for rows of 2 KB and less (16384 x 1024 fp16: 33 -> 23 us); with more rows than waves a
    // wave walks several rows and the waves of a CU drift apart
    const int64_t row_bytes = cols * (int64_t)sizeof(S);
    int64_t per_cu = 32768 / row_bytes;
    per_cu = per_cu < 4 ? 4 : (per_cu > 16 ? 16 : per_cu);
    const int64_t wcap = 256 * per_cu;
    const int64_t waves = rows < wcap ? rows : wcap;
    const int grid = (int)((waves + kWavesPerBlock - 1) / kWavesPerBlock);
    nparts = (int64_t)grid * kWavesPerBlock < rows ? (int64_t)grid * kWavesPerBlock : rows;
#define OFQ_LN_WAVE(NPV)                                                                       \
  ln_observer_wave_rows<T, NPV, SKIP, EXACT><<<grid, kLnBlock, 0, st>>>(xs, gs, bs, ys, ws, rows, \
                                                                        cols, eps, sk)
    if (npacks <= kWave) {
      OFQ_LN_WAVE(1);
    } else if (npacks <= 2 * kWave) {
      OFQ_LN_WAVE(2);
    } else if (npacks <= 4 * kWave) {
      OFQ_LN_WAVE(4);
    } else {
      OFQ_LN_WAVE(8);
    }
#undef OFQ_LN_WAVE
  } else if (vec_ok && npacks <= kLnBlock) {
    ln_observer_rows<T, 1, SKIP, EXACT><<<(int)rows, kLnBlock, 0, st>>>(xs, gs, bs, ys, ws, cols, eps, sk);
  } else if (vec_ok && npacks <= 2 * kLnBlock) {
    ln_observer_rows<T, 2, SKIP, EXACT><<<(int)rows, kLnBlock, 0, st>>>(xs, gs, bs, ys, ws, cols, eps, sk);
  } else if (vec_ok && npacks <= 4 * kLnBlock) {
    ln_observer_rows<T, 4, SKIP, EXACT><<<(int)rows, kLnBlock, 0, st>>>(xs, gs, bs, ys, ws, cols, eps, sk);
  } else if (vec_ok && npacks <= 8 * kLnBlock) {
    ln_observer_rows<T, 8, SKIP, EXACT><<<(int)rows, kLnBlock, 0, st>>>(xs, gs, bs, ys, ws, cols, eps, sk);
  } else {
    ln_observer_rows_generic<T, SKIP, EXACT><<<(int)rows, kLnBlock, 0, st>>>(xs, gs, bs, ys, ws, cols,
                                                                      eps, sk);
  }
  ln_observer_finalize<<<1, ln_final_threads(nparts), 0, st>>>(ws, nparts, bits, scale, zero_point);
  return ofq_check_launch();
}

int run(void* stream, const void* x, const void* bias, const void* skip, double alpha,
        bool with_skip, const void* gamma, const void* beta, void* y, float* scale,
        float* zero_point, int t_dtype, int64_t rows, int64_t cols, double epsilon,
        int quantization_bit, int statistics, void* workspace, size_t workspace_bytes) {
  OFQ_RETURN_IF(quantization_bit <= 1 || quantization_bit > 8, OFQ_ERR_BAD_ATTR);
  OFQ_RETURN_IF(statistics != OFQ_LN_STATS_FP32 && statistics != OFQ_LN_STATS_FP64,
                OFQ_ERR_BAD_ATTR);
  OFQ_RETURN_IF(t_dtype != OFQ_F16 && t_dtype != OFQ_BF16 && t_dtype != OFQ_F32,
                OFQ_ERR_BAD_DTYPE);
  OFQ_RETURN_IF(rows < 1 || cols < 1 || rows > 0x7FFFFFFF, OFQ_ERR_BAD_SHAPE);
  OFQ_RETURN_IF(x == nullptr || y == nullptr || scale == nullptr || zero_point == nullptr,
                OFQ_ERR_NULL_POINTER);
  OFQ_RETURN_IF(workspace == nullptr || workspace_bytes < (size_t)rows * sizeof(float),
                OFQ_ERR_WORKSPACE);
  hipStream_t st = static_cast<hipStream_t>(stream);
  float* ws = static_cast<float*>(workspace);
  const double eps = epsilon;  // (the fp32 statistics round it to fp32 in the kernel)
#define OFQ_LN_RUN2(T, EX)                                                                     \
  return with_skip ? launch<T, true, EX>(st, x, gamma, beta, y, scale, zero_point, rows, cols, \
                                         eps, quantization_bit, ws, bias, skip, alpha)         \
                   : launch<T, false, EX>(st, x, gamma, beta, y, scale, zero_point, rows,      \
                                          cols, eps, quantization_bit, ws, nullptr, nullptr, 0.0)
#define OFQ_LN_RUN(T)                                    \
  if (statistics == OFQ_LN_STATS_FP64) OFQ_LN_RUN2(T, true); \
  OFQ_LN_RUN2(T, false)
  switch (t_dtype) {
    case OFQ_F16: OFQ_LN_RUN(f16);
    case OFQ_BF16: OFQ_LN_RUN(bf16);
    default: OFQ_LN_RUN(float);
  }
#undef OFQ_LN_RUN
#undef OFQ_LN_RUN2
}

// device address of `scratch` on the current device, looked up once per device
constexpr int kMaxDevices = 64;
std::atomic<float*> scratch_on_device[kMaxDevices];

int static_scratch(float** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return OFQ_ERR_LAUNCH;
  float* p = scratch_on_device[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    void* addr = nullptr;
    if (hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch)) != hipSuccess || addr == nullptr) {
      return OFQ_ERR_LAUNCH;
    }
    p = static_cast<float*>(addr);
    scratch_on_device[dev].store(p, std::memory_order_release);  // same value from any thread
  }
  *out = p;
  return OFQ_OK;
}

}  // namespace
}  // namespace ofq

extern "C" int ofq_fused_layer_norm_min_max_observer_static(void* stream, const void* x,
                                                            const void* gamma, const void* beta,
                                                            void* y, float* scale,
                                                            float* zero_point, int t_dtype,
                                                            int64_t rows, int64_t cols,
                                                            double epsilon, int quantization_bit) {
  if (rows > OFQ_LN_STATIC_MAX_ROWS) return OFQ_ERR_TOO_LARGE;
  float* ws = nullptr;
  const int st = ofq::static_scratch(&ws);
  if (st != OFQ_OK) return st;
  // every partial the finalize kernel reads is written by the row kernel of the same call, so
  // nothing has to be cleared between calls
  return ofq::run(stream, x, nullptr, nullptr, 0.0, false, gamma, beta, y, scale, zero_point,
                  t_dtype, rows, cols, epsilon, quantization_bit, OFQ_LN_STATS_FP32, ws,
                  (size_t)OFQ_LN_STATIC_MAX_ROWS * sizeof(float));
}

extern "C" size_t ofq_fused_layer_norm_min_max_observer_workspace_bytes(int, int64_t rows,
                                                                        int64_t) {
  return rows > 0 ? (size_t)rows * sizeof(float) : 0;
}

extern "C" int ofq_fused_layer_norm_min_max_observer(void* stream, const void* x,
                                                     const void* gamma, const void* beta, void* y,
                                                     float* scale, float* zero_point, int t_dtype,
                                                     int64_t rows, int64_t cols, double epsilon,
                                                     int quantization_bit, void* workspace,
                                                     size_t workspace_bytes) {
  return ofq::run(stream, x, nullptr, nullptr, 0.0, false, gamma, beta, y, scale, zero_point,
                  t_dtype, rows, cols, epsilon, quantization_bit, OFQ_LN_STATS_FP32, workspace,
                  workspace_bytes);
}

extern "C" int ofq_fused_skip_layer_norm_min_max_observer(
    void* stream, const void* x, const void* bias, const void* skip, double alpha,
    const void* gamma, const void* beta, void* y, float* scale, float* zero_point, int t_dtype,
    int64_t rows, int64_t cols, double epsilon, int quantization_bit, void* workspace,
    size_t workspace_bytes) {
  return ofq::run(stream, x, bias, skip, alpha, true, gamma, beta, y, scale, zero_point, t_dtype,
                  rows, cols, epsilon, quantization_bit, OFQ_LN_STATS_FP32, workspace,
                  workspace_bytes);
}


namespace ofq {
namespace {

template<typename T, bool EXACT>
void launch_ln_quant_any(hipStream_t st, const LnQuantArgs& a) {
  const int packs = a.cols / 8;
  if (a.rows <= ln_one_block_rows<T>(packs, kLnCodes)) ln_one_block<T, EXACT, kLnCodes, false>(st, a, LnSkip16{});
  else if (packs <= kWave) launch_ln_quant_rows<T, 1, 1, EXACT>(st, a);
  else if (packs <= 2 * kWave) launch_ln_quant_rows<T, 2, 1, EXACT>(st, a);
  else if (packs <= 4 * kWave) launch_ln_quant_rows<T, 4, 1, EXACT>(st, a);
  else if (packs <= 8 * kWave) launch_ln_quant_rows<T, 8, 1, EXACT>(st, a);
  else if (packs <= 16 * kWave) launch_ln_quant_rows<T, 4, 4, EXACT>(st, a);
  else launch_ln_quant_rows<T, 8, 4, EXACT>(st, a);
}

// the shapes ln_quant_first and ln_quant_second take
bool ln_quant_full(const void* x, const void* gamma, const void* beta, const void* codes, int t_dtype,
                   int64_t cols) {
  const int64_t np = cols / 512;
  return t_dtype == OFQ_F16 && gamma != nullptr && beta != nullptr && cols % 512 == 0
         && (np == 1 || np == 2 || np == 4 || np == 8) && ofq_aligned16(x) && ofq_aligned16(gamma)
         && ofq_aligned16(beta) && (reinterpret_cast<uintptr_t>(codes) & 7u) == 0;
}

}  // namespace
}  // namespace ofq

extern "C" size_t ofq_fused_layer_norm_quantization_workspace_bytes(int, int64_t rows, int64_t) {
  // [partial maxima: rows floats, padded to 16 bytes][(mean, inv) of every row]
  return rows > 0 ? (((size_t)rows * sizeof(float) + 15) & ~(size_t)15) + (size_t)rows * 2 * sizeof(float)
                  : 0;
}

namespace ofq {
namespace {

int ln_quant(void* stream, const void* x, const void* gamma, const void* beta, void* codes, float* scale,
             float* zero_point, int t_dtype, int64_t rows, int64_t cols, double epsilon, int quantization_bit,
             int statistics, void* workspace, size_t workspace_bytes, bool any_row) {
  OFQ_RETURN_IF(quantization_bit <= 1 || quantization_bit > 8, OFQ_ERR_BAD_ATTR);
  OFQ_RETURN_IF(statistics != OFQ_LN_STATS_FP32 && statistics != OFQ_LN_STATS_FP64,
                OFQ_ERR_BAD_ATTR);
  OFQ_RETURN_IF(t_dtype != OFQ_F16 && t_dtype != OFQ_BF16 && t_dtype != OFQ_F32,
                OFQ_ERR_BAD_DTYPE);
  OFQ_RETURN_IF(rows < 1 || cols < 1 || rows > 0x7FFFFFFF, OFQ_ERR_BAD_SHAPE);
  OFQ_RETURN_IF(x == nullptr || codes == nullptr || scale == nullptr || zero_point == nullptr,
                OFQ_ERR_NULL_POINTER);
  OFQ_RETURN_IF(workspace == nullptr
                    || workspace_bytes
                           < ofq_fused_layer_norm_quantization_workspace_bytes(t_dtype, rows, cols)
                    || !ofq_aligned16(workspace),
                OFQ_ERR_WORKSPACE);
  // the shapes the register-resident row kernels take; everything else is the two ops in a row
  const bool full = ln_quant_full(x, gamma, beta, codes, t_dtype, cols);
  const bool rows8 = t_dtype != OFQ_F32 && cols % 8 == 0 && cols <= 16384 && ofq_aligned16(x)
                     && ofq_aligned16(gamma) && ofq_aligned16(beta)
                     && (reinterpret_cast<uintptr_t>(codes) & 7u) == 0;
  OFQ_RETURN_IF(!(full || (any_row && rows8)), OFQ_ERR_UNSUPPORTED);
  hipStream_t st = static_cast<hipStream_t>(stream);
  float* part = static_cast<float*>(workspace);
  float* stats = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace)
                                          + (((size_t)rows * sizeof(float) + 15) & ~(size_t)15));
  const uint16_t* xs = static_cast<const uint16_t*>(x);
  const uint16_t* gs = static_cast<const uint16_t*>(gamma);
  const uint16_t* bs = static_cast<const uint16_t*>(beta);
  const bool exact = statistics == OFQ_LN_STATS_FP64;
  const int np = (int)(cols / 512);
  const LnQuantArgs args = {xs, gs, bs, part, stats, codes, scale, zero_point, rows,
                            (int)cols, epsilon, quantization_bit};
  if (!full) {
    if (t_dtype == OFQ_F16) {
      if (exact) launch_ln_quant_any<f16, true>(st, args);
      else launch_ln_quant_any<f16, false>(st, args);
    } else {
      if (exact) launch_ln_quant_any<bf16, true>(st, args);
      else launch_ln_quant_any<bf16, false>(st, args);
    }
    return ofq_check_launch();
  }
  if (rows <= ln_one_block_rows<f16>((int)(cols / 8), kLnCodes)) {
    if (exact) ln_one_block<f16, true, kLnCodes, false>(st, args, LnSkip16{});
    else ln_one_block<f16, false, kLnCodes, false>(st, args, LnSkip16{});
    return ofq_check_launch();
  }
  // one row per wave up to 16 waves per CU, beyond that the waves walk the rows; both kernels
  // use the same grid, so a row meets the same wave of the same block twice
  const int64_t waves = rows < 256 * 16 ? rows : 256 * 16;
  constexpr int kWavesPerBlock = kLnqBlock / kWave;
  const int grid = (int)((waves + kWavesPerBlock - 1) / kWavesPerBlock);
  const int64_t nparts = grid;  // one partial maximum per block of the first kernel (<= 512)
  // parts of a row in the second kernel: enough waves for 16 per CU where the rows allow it
  int split = 1;
  while (split < 4 && split * 2 <= np && waves * split * 2 <= 256 * 16) split *= 2;
  const int grid2 = (grid + 7) / 8 * 8 * split;
#define OFQ_LNQ1(NPV)                                                                           \
  if (exact) {                                                                                  \
    ln_quant_first<NPV, true><<<grid, kLnqBlock, 0, st>>>(xs, gs, bs, part, stats, rows, epsilon);  \
  } else {                                                                                      \
    ln_quant_first<NPV, false><<<grid, kLnqBlock, 0, st>>>(xs, gs, bs, part, stats, rows, epsilon); \
  }
#define OFQ_LNQ2(NPV, SPV)                                                                      \
  if (split == SPV) {                                                                           \
    ln_quant_second<NPV, SPV><<<grid2, kLnqBlock, 0, st>>>(                                     \
        xs, gs, bs, part, nparts, stats, static_cast<int8_t*>(codes), scale, zero_point, rows,  \
        quantization_bit, grid);                                                                \
  }
  switch (np) {
    case 1: OFQ_LNQ1(1) OFQ_LNQ2(1, 1) break;
    case 2: OFQ_LNQ1(2) OFQ_LNQ2(2, 1) OFQ_LNQ2(2, 2) break;
    case 4: OFQ_LNQ1(4) OFQ_LNQ2(4, 1) OFQ_LNQ2(4, 2) OFQ_LNQ2(4, 4) break;
    default: OFQ_LNQ1(8) OFQ_LNQ2(8, 1) OFQ_LNQ2(8, 2) OFQ_LNQ2(8, 4) break;
  }
#undef OFQ_LNQ1
#undef OFQ_LNQ2
  return ofq_check_launch();
}

}  // namespace
}  // namespace ofq

extern "C" int ofq_fused_layer_norm_quantization(void* stream, const void* x, const void* gamma,
                                                 const void* beta, void* codes, float* scale,
                                                 float* zero_point, int t_dtype, int64_t rows,
                                                 int64_t cols, double epsilon, int quantization_bit,
                                                 int statistics, void* workspace,
                                                 size_t workspace_bytes) {
  return ofq::ln_quant(stream, x, gamma, beta, codes, scale, zero_point, t_dtype, rows, cols, epsilon,
                       quantization_bit, statistics, workspace, workspace_bytes, false);
}

extern "C" int ofq_fused_layer_norm_quantization_any_row(
    void* stream, const void* x, const void* gamma, const void* beta, void* codes, float* scale,
    float* zero_point, int t_dtype, int64_t rows, int64_t cols, double epsilon, int quantization_bit,
    int statistics, void* workspace, size_t workspace_bytes) {
  return ofq::ln_quant(stream, x, gamma, beta, codes, scale, zero_point, t_dtype, rows, cols, epsilon,
                       quantization_bit, statistics, workspace, workspace_bytes, true);
}

extern "C" int ofq_fused_layer_norm_min_max_observer_stats(
    void* stream, const void* x, const void* bias, const void* skip, double alpha, int with_skip,
    const void* gamma, const void* beta, void* y, float* scale, float* zero_point, int t_dtype,
    int64_t rows, int64_t cols, double epsilon, int quantization_bit, int statistics,
    void* workspace, size_t workspace_bytes) {
  return ofq::run(stream, x, with_skip ? bias : nullptr, with_skip ? skip : nullptr,
                  with_skip ? alpha : 0.0, with_skip != 0, gamma, beta, y, scale, zero_point,
                  t_dtype, rows, cols, epsilon, quantization_bit, statistics, workspace,
                  workspace_bytes);
}
