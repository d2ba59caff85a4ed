// The second pass of a K split.
#pragma once

#include "common.h"
#include "gelu.h"

namespace ferrite {
namespace {

// out = sum over the K slices of the f32 partial slabs, in slice order
// (deterministic), cast to TO. The slabs are `slab` floats apart (slab % 4 == 0, slab >= mn);
// the GELU epilogues need mn % 4 == 0.
template <typename TO, int EPI = kEpiNone>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float* __restrict__ part, TO* __restrict__ out,
                                                                int64_t mn, int slices, bf16* __restrict__ aux,
                                                                int64_t slab) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= mn) return;
  f32x4 acc = *reinterpret_cast<const f32x4*>(part + i);
  for (int s = 1; s < slices; ++s) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(part + (int64_t)s * slab + i);
    acc += v;
  }
  if (EPI == kEpiNone && i + 4 > mn) {
    for (int e = 0; e < (int)(mn - i); ++e) out[i + e] = Elem<TO>::from_f32(acc[e]);
    return;
  }
  if constexpr (EPI != kEpiNone)
    gelu_epilogue<EPI>(bf16x4{(bf16)acc[0], (bf16)acc[1], (bf16)acc[2], (bf16)acc[3]}, reinterpret_cast<bf16*>(out + i),
                       aux + i);
  else if constexpr (sizeof(TO) == 2)
    *reinterpret_cast<bf16x4*>(out + i) = bf16x4{(bf16)acc[0], (bf16)acc[1], (bf16)acc[2], (bf16)acc[3]};
  else
    *reinterpret_cast<f32x4*>(out + i) = acc;
}

}  // namespace
}  // namespace ferrite
