// Products of few rows (skinny.hip): out[M,N] = x[M,K] . w with M <= kSkinnyRows.
#pragma once

#include "common.h"

namespace ferrite {

// Rows up to which the skinny kernels take a product: two 32-row MFMA blocks.
constexpr int64_t kSkinnyRows = 64;

// x bf16 [M,K]; w [K,N] (or, w_t, [N,K]) bf16, or float whose elements are rounded to bf16 as
// they are read; out f32 or bf16 by out_dtype. epi: kEpiNone, kEpiGelu (a float w: not
// transposed) or kEpiGeluGrad (bf16 w) of gelu.h with a bf16 out and aux. Any sizes and
// element-aligned pointers.
struct SkinnyArgs {
  const void* x;
  const void* w;
  void* out;
  void* aux;
  int64_t m, n, k;
  bool w_t;
  int w_dtype, out_dtype, epi;
  void* ws;  // f32 partials of a K split, or nullptr
  int64_t ws_bytes;
};
// Sizes the kernels take.
bool skinny_ok(int64_t m, int64_t n, int64_t k);
// Of those, where they beat the 256-row tiles for operands that both read in place: up to 2^24
// weights, and beyond for a few rows and a deep K. The tiles' time does not depend on M, the
// skinny kernels read x again in every workgroup (us on one MI355X, skinny / tiles):
// M = 64: 4096 x 4096 19.2 / 21.8, 8192 x 8192 50 / 41, 768 x 32768 24 / 14;
// M = 8: 8192 x 8192 35 / 38, 768 x 32768 14.4 / 13.0.
bool skinny_better(int64_t m, int64_t n, int64_t k);
// Bytes of the K split's partials, 0 where there is none; without them K is not split.
int64_t skinny_workspace(const SkinnyArgs& a);
int skinny_launch(const SkinnyArgs& a, hipStream_t stream);

}  // namespace ferrite
