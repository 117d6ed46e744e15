// Launchers shared between translation units of the library (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ofq {

struct LinearArgs {
  const void* x;        // [m,k] T
  const void* w;        // [n, k*bits/8] bytes
  const void* scale;    // [n, k/group_size] T
  const void* zero;     // same or nullptr
  const void* bias;     // [n] T or nullptr
  void* out;            // [m,n] T
  int t_dtype;          // OFQ_F16 | OFQ_BF16 | OFQ_F32
  bool w_signed;        // int8 container
  int bits;             // 4 | 8
  bool symmetric;
  int group_dim;        // 0 | 1
  int64_t group_size;
  int64_t m, n, k;
};

// MFMA GEMM with in-tile dequantisation; groups along K.  Returns OFQ_ERR_UNSUPPORTED when the
// shape does not meet the kernel's tiling constraints (caller falls back).
// With a workspace of gemm_wq_workspace_bytes() K is cut into slices where the tiles do not fill the chip, or,
// from 1024 rows on and where that is expected to take less, the weight is dequantised once into it and a copy-fed GEMM
// runs on the result; without one a block walks all of K, on packed weights.
bool gemm_wq_supported(const LinearArgs& a);
size_t gemm_wq_workspace_bytes(const LinearArgs& a);
int launch_gemm_wq(hipStream_t st, const LinearArgs& a, void* workspace, size_t workspace_bytes);

// The GEMM whose weights stay packed until they are in registers (gemm_wr.h): a tile of rows of x by
// columns of the output and a number of K slices.
enum WrTile { kWr32x128, kWr64x128, kWr96x128, kWr128x256, kWr192x256 };
struct WrPlan {
  WrTile tile;
  int splits;
};
// the plan that launch_gemm_wq takes with a workspace of gemm_wq_workspace_bytes() or without one (then of
// one slice); false: not this kernel's problem
bool gemm_wr_plan(const LinearArgs& a, bool have_workspace, WrPlan* plan);
// expected time (us; 1e30: not this kernel's problem) of a problem of 16 < m <= 64 on it, with two_launches
// added if it takes two
double gemm_wr_us(const LinearArgs& a, bool have_workspace, double two_launches);
int launch_gemm_wr_f16(hipStream_t st, const LinearArgs& a, const WrPlan& plan, float* partials);
int launch_gemm_wr_bf16(hipStream_t st, const LinearArgs& a, const WrPlan& plan, float* partials);

// Copy-fed GEMMs for more than 128 rows (gemm_pp.h) on tiles of 256 x width (384, 256 or 192; rows that are
// not a multiple of 128 bytes 384 only, or 256 in int8); the linear's with the weight already in the dtype
// of x.
int launch_gemm_pp_f16(hipStream_t st, const void* x, const void* w, const void* bias, void* out,
                       int64_t m, int64_t n, int64_t k, int width);
int launch_gemm_pp_bf16(hipStream_t st, const void* x, const void* w, const void* bias, void* out,
                        int64_t m, int64_t n, int64_t k, int width);
int launch_gemm_pp_i8(hipStream_t st, const void* a, const void* b, const float* a_scale,
                      const float* b_scale, const void* bias, void* out, int out_dtype, int64_t m,
                      int64_t n, int64_t k, int width);

// m = 1, fp16, 4-bit symmetric codes in an int8 container, groups along K: a wave owns whole
// weight rows (contiguous requests, packed dot products, no cross-wave fold).
bool gemv_m1_supported(const LinearArgs& a);
int launch_gemv_m1(hipStream_t st, const LinearArgs& a);
int launch_gemv_m1_grouped(hipStream_t st, const LinearArgs* problems, int count);
int launch_gemv_m1_glu(hipStream_t st, const LinearArgs& a, const LinearArgs& g, void* y, int act);
// the same for groups along N (scale [n / group_size, k]): the scale meets x, once per block
bool gemv_m1_gn_supported(const LinearArgs& a);
int launch_gemv_m1_gn(hipStream_t st, const LinearArgs& a);

// m = 1, fp16 or bf16, 4- or 8-bit codes in either container, symmetric or with a zero point,
// groups along K of a power-of-two size: the same row-per-wave structure with the reference's
// roundings of w~.
bool gemv_m1_any_supported(const LinearArgs& a);
int launch_gemv_m1_any(hipStream_t st, const LinearArgs& a);

// Skinny-M (m <= 16) MFMA GEMV that streams the weights once.
bool gemv_wq_supported(const LinearArgs& a);
int launch_gemv_wq(hipStream_t st, const LinearArgs& a);

// 16 < m <= 64: the streaming kernels with several 16-row tiles of x per weight tile, without a
// workspace.  Not where gemm_wr is expected to take less; `choice` is which of the two runs, and how.
struct MtChoice;
bool gemv_mt_preferred(const LinearArgs& a, bool have_workspace, MtChoice* choice);
int launch_gemv_mt(hipStream_t st, const LinearArgs& a, const MtChoice& choice);
// several of them, or a gated unit's two with y = out0 * act(out1), in one launch where that is expected to
// take less than one by one; else OFQ_ERR_UNSUPPORTED
int launch_gemv_mt_several(hipStream_t st, const LinearArgs* problems, int count, bool glu, void* y, int act);

// Groups along N (group_dim = 0), fp16 / bf16: the streaming kernel with one scale per k (any m,
// 64 rows of x per pass over the weights), and for m > 64 with a workspace of
// gemm_gn_workspace_bytes() the weight dequantised once plus a copy-fed GEMM.
bool gemv_gn_supported(const LinearArgs& a);
int launch_gemv_gn(hipStream_t st, const LinearArgs& a);
size_t gemm_gn_workspace_bytes(const LinearArgs& a);
int launch_gemm_gn(hipStream_t st, const LinearArgs& a, void* workspace);

// Up to 8 decode linears that share m, k, dtype and quantisation attributes (x, w, scale, zero,
// bias, out and n per problem) as ONE launch of the natural-order decode kernel.
// OFQ_ERR_UNSUPPORTED when the shapes do not fit it (caller launches the problems one by one).
int launch_gemv_grouped(hipStream_t st, const LinearArgs* problems, int count);

// fused_glu in split mode for decode: hidden = x w~^T + b -> a.out, gate = x v~^T + c -> g.out,
// y = hidden * act(gate), all in ONE launch (every block owns the same rows of both weights).
// a and g differ in w / scale / zero / bias / out only.  OFQ_ERR_UNSUPPORTED when the shapes do
// not fit (caller runs the linears and the gating separately).
int launch_gemv_glu(hipStream_t st, const LinearArgs& a, const LinearArgs& g, void* y, int act);

// What one launch of a streaming kernel works on: one linear, several that share m, k, dtype and quantisation
// attributes, or the two of a gated unit (problems 0 and 1 of equal n and x, then y = out0 * act(out1)).
struct LinearJob {
  const LinearArgs* pr;
  int count;
  bool glu;
  void* y;
  int act;
};
// The ring kernel (gemv_ring.h), up to 16 rows of x
struct RingPlan {
  int grid, rows_per_block, tr, tl, wk_shift, phase_steps, phases;
  size_t lds;
};
bool gemv_ring_choice(const LinearJob& job, RingPlan* plan);
int launch_gemv_ring_f16(hipStream_t st, const LinearJob& job, const RingPlan& plan);
int launch_gemv_ring_bf16(hipStream_t st, const LinearJob& job, const RingPlan& plan);
// The kernel whose waves share nothing (gemv_flow.h), up to 48 rows of x; the choice: up to 16
struct FlowPlan {
  int grid, rows_per_block, mx, tl, nw;
  int tiled;  // the weight is its tile-major copy
  size_t lds;
};
bool gemv_flow_choice(const LinearJob& job, FlowPlan* plan);
int launch_gemv_flow_f16_b4(hipStream_t st, const LinearJob& job, const FlowPlan& plan);
int launch_gemv_flow_f16_b8(hipStream_t st, const LinearJob& job, const FlowPlan& plan);
int launch_gemv_flow_bf16_b4(hipStream_t st, const LinearJob& job, const FlowPlan& plan);
int launch_gemv_flow_bf16_b8(hipStream_t st, const LinearJob& job, const FlowPlan& plan);
// gemv_rows_mt (gemv_rows.h), 17 to 64 rows of x
struct RowsMtPlan {
  int grid, rows_per_block, panel_chunks, panel_groups;
  size_t lds;
};
int launch_gemv_mt_f16(hipStream_t st, const LinearJob& job, const RowsMtPlan& plan);
int launch_gemv_mt_bf16(hipStream_t st, const LinearJob& job, const RowsMtPlan& plan);
// gemv_ring_mt (gemv_ring_mt.h), 17 to 64 rows of x
struct RingMtPlan {
  int grid, rows_per_block, tl, wk, depth, buffers, phases;
  size_t lds;
};
// the faster of the two for a job, and its expected time
struct MtChoice {
  bool ring;  // gemv_ring_mt, by `plan`
  RingMtPlan plan;
  double us;
};
void gemv_mt_choice(const LinearJob& job, MtChoice* choice);
int launch_gemv_ring_mt_f16_b4(hipStream_t st, const LinearJob& job, const RingMtPlan& plan);
int launch_gemv_ring_mt_f16_b8(hipStream_t st, const LinearJob& job, const RingMtPlan& plan);
int launch_gemv_ring_mt_bf16_b4(hipStream_t st, const LinearJob& job, const RingMtPlan& plan);
int launch_gemv_ring_mt_bf16_b8(hipStream_t st, const LinearJob& job, const RingMtPlan& plan);

// matmul_quant with few rows of a (m <= 96; k a multiple of 64): int8 MFMA with the weights
// streamed once; its expected time (m > 64).
double matmul_quant_rows_us(int64_t m, int64_t n, int64_t k);
bool matmul_quant_rows_supported(int64_t m, int64_t n, int64_t k);
int launch_matmul_quant_rows(hipStream_t st, const void* a, const void* b, const float* a_scale,
                             const float* b_scale, const void* bias, void* out, int out_dtype,
                             int64_t m, int64_t n, int64_t k);

// Any shape / grouping; one wave per output element.
int launch_linear_generic(hipStream_t st, const LinearArgs& a);

}  // namespace ofq
