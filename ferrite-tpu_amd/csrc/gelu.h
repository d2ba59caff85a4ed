// The tanh GELU and its derivative as the matmul epilogues apply them (the MLP of
// model/gpt.py:141: jax.nn.gelu(approximate=True)).
//
// gelu(u) = u/2 (1 + tanh(z)), z = b (u + c u^3), b = sqrt(2/pi), c = 0.044715,
// written as u s with s = (1 + tanh z)/2 = 1 / (1 + 2^(-2 z log2 e)): one exp2
// and one reciprocal instead of a libm tanh (the epilogue runs once per output
// element, after the products, with nothing to hide it behind), and no
// cancellation in 1 + tanh z at negative u. gelu'(u) = s + 2 u s (1 - s) b (1 + 3 c u^2).
// Both in f32 from the bf16-rounded u, as an elementwise pass over the rounded
// product computes them.

#pragma once

#include "common.h"

namespace ferrite {
namespace {

constexpr int kEpiNone = 0, kEpiGelu = 1, kEpiGeluGrad = 2;
constexpr float kGeluB = 0.7978845608028654f, kGeluC = 0.044715f;
constexpr float kGeluE = -2.0f * kGeluB * 1.4426950408889634f;  // -2 b log2(e)

__device__ __forceinline__ float gelu_gate(float u) {  // s = (1 + tanh z) / 2
  return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(kGeluE * (u + kGeluC * u * u * u)));
}
__device__ __forceinline__ float gelu_tanh(float u) { return u * gelu_gate(u); }
__device__ __forceinline__ float gelu_tanh_grad(float u) {
  const float s = gelu_gate(u);
  return s + 2.f * u * s * (1.f - s) * kGeluB * (1.f + 3.f * kGeluC * u * u);
}

// Four consecutive outputs v = bf16(x . y) of one row. kEpiGelu: aux <- v (the
// pre-activation), out <- bf16(gelu(v)). kEpiGeluGrad: u is the pre-activation
// (read from aux); out <- bf16(v * gelu'(u)) (v is the incoming gradient).
__device__ __forceinline__ void gelu_store(const bf16x4& v, bf16* out, bf16* aux) {
  *reinterpret_cast<bf16x4*>(aux) = v;
  bf16x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = (bf16)gelu_tanh((float)v[e]);
  *reinterpret_cast<bf16x4*>(out) = r;
}
__device__ __forceinline__ void gelu_grad_store(const bf16x4& v, const bf16x4& u, bf16* out) {
  bf16x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = (bf16)((float)v[e] * gelu_tanh_grad((float)u[e]));
  *reinterpret_cast<bf16x4*>(out) = r;
}
template <int EPI>
__device__ __forceinline__ void gelu_epilogue(const bf16x4& v, bf16* out, bf16* aux) {
  if constexpr (EPI == kEpiGelu)
    gelu_store(v, out, aux);
  else
    gelu_grad_store(v, *reinterpret_cast<const bf16x4*>(aux), out);
}

}  // namespace
}  // namespace ferrite
