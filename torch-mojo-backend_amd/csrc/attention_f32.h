// f32 attention on matrix cores (attention_f32.hip), behind the entry points
// of attention_generic.hip.
#pragma once
#include "common.h"

namespace mi {

// Operands with (batch, head, row) strides and a unit head-dim stride.
struct AttnF32 {
  float* o; int64_t o_b, o_h, o_s;
  float* lse;
  const float* q; int64_t q_b, q_h, q_s;
  const float* k; int64_t k_b, k_h, k_s;
  const float* v; int64_t v_b, v_h, v_s;
  const float* dout; int64_t do_b, do_h, do_s;
  float* dq; int64_t dq_b, dq_h, dq_s;
  float* dk; int64_t dk_b, dk_h, dk_s;
  float* dv; int64_t dv_b, dv_h, dv_s;
  float* delta;  // [B, H, Sq]
  int64_t B, H, Sq, Skv;
  float scale_log2, scale;  // scale * log2(e), scale
  int causal;
};

// -1 when the inputs are not taken (other head dims, unaligned rows).
int attn_f32_fwd(const AttnF32& p, int64_t d, hipStream_t s);
int attn_f32_bwd(const AttnF32& p, int64_t d, hipStream_t s);

}  // namespace mi
