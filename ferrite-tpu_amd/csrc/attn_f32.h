// Attention in float32 (attn_f32.hip): head dims up to 128 with 16-byte aligned rows.
#pragma once

#include "common.h"

namespace ferrite {

// Dense [b h, sq, d] and [b h, sk, d] tensors, d <= 128 and d % 4 == 0.
struct F32Attn {
  int64_t bh, sq, sk, d;
  int causal;
};
int f32_attn_fwd(const float* q, const float* k, const float* v, float* o, float* lse, const F32Attn& s, float scale,
                 hipStream_t stream);
int f32_attn_dq(const float* q, const float* k, const float* v, const float* dout, const float* lse, const float* delta,
                float* dq, const F32Attn& s, float scale, hipStream_t stream);
int f32_attn_dkv(const float* q, const float* k, const float* v, const float* dout, const float* lse,
                 const float* delta, float* dk, float* dv, const F32Attn& s, float scale, hipStream_t stream);

}  // namespace ferrite
