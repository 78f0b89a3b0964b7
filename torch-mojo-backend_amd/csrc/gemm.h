// What the GEMM kernels share: one call's arguments, element access by dtype
// code, and the sum of split-K partials.
#pragma once
#include "common.h"

namespace mi {

struct GemmArgs {
  void* c;
  int c_dt;
  int64_t c_rs, c_bs;
  const void* a;
  int64_t a_rs, a_cs, a_bs;
  const void* b;
  int64_t b_rs, b_cs, b_bs;
  const void* bias;
  int bias_dt;
  int beta;
  int64_t m, n, k;
  float* part;     // split-K partials [splits][batch][m][n] (f32) or null
  int64_t kchunk;  // K per split
  int tiles_n;     // tiles along n
  int group;       // tile rows walked together (1: row by row)
  int batch;       // batch count (grid.y = splits * batch)
  int ab_dt;       // operand dtype (for rounding through it)
  int round_c;     // round C (and the row sums) through ab_dt before storing
  void* rowsum;    // optional sum over k of A's rows [batch][m], or null
  int rowsum_dt;
  float* rs_part;  // split-K row-sum partials [splits * rs_slots][batch][m]
};

// v rounded to the 16-bit operand dtype and widened back.
__device__ __forceinline__ float round_through(float v, int dt) {
  return dt == MI355X_BF16 ? (float)(bf16)v : (float)(f16)v;
}

__device__ __forceinline__ float ld_any(const void* p, int dt, int64_t i) {
  switch (dt) {
    case MI355X_F32: return ((const float*)p)[i];
    case MI355X_BF16: return (float)((const bf16*)p)[i];
    default: return (float)((const f16*)p)[i];
  }
}
__device__ __forceinline__ void st_any(void* p, int dt, int64_t i, float v) {
  switch (dt) {
    case MI355X_F32: ((float*)p)[i] = v; break;
    case MI355X_BF16: ((bf16*)p)[i] = (bf16)v; break;
    default: ((f16*)p)[i] = (f16)v; break;
  }
}

// C = sum of the split-K partials (+ bias) (+ C), launched on `s`; with
// rs_slots > 0 the row sums too.  Returns -1 when C is done by the scalar
// kernel, which leaves the row sums to the caller.
int splitk_finish(const GemmArgs& g, int64_t batch, int splits, int rs_slots, hipStream_t s);

// One launch of the 16-bit MFMA tiles (gemm_tile.h) in block configuration
// `cfg`; KT: K is not a multiple of 64.
template <typename T, bool KT>
int gemm_tiles(const GemmArgs& g, int64_t batch, int cfg, int splits, hipStream_t s);
extern template int gemm_tiles<bf16, false>(const GemmArgs&, int64_t, int, int, hipStream_t);
extern template int gemm_tiles<bf16, true>(const GemmArgs&, int64_t, int, int, hipStream_t);
extern template int gemm_tiles<f16, false>(const GemmArgs&, int64_t, int, int, hipStream_t);
extern template int gemm_tiles<f16, true>(const GemmArgs&, int64_t, int, int, hipStream_t);

// f32 operands (gemm_f32.hip): bytes of split-K partials that the call can
// use, and the launch, which runs without splits when it has no workspace.
int64_t gemm_f32_workspace(int64_t batch, int64_t m, int64_t n, int64_t k);
int gemm_f32_launch(GemmArgs g, int64_t batch, void* workspace, int64_t ws_bytes, hipStream_t s);

}  // namespace mi
