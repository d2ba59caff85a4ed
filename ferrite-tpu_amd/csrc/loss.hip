// Softmax cross-entropy over f32 logits, for gfx950.
//
// Reference: src/ferrite/model/gpt.py:147-152 (loss_fn: log_softmax in f32,
// negative log-likelihood of the target, mean over tokens) and its autodiff
// backward, d logits = (softmax - onehot(target)) * dloss / N.
//
// HBM-bound on the [N, V] logits (1 GiB at N = 8192, V = 32768): the forward
// reads them once, keeping an online (max, sum of exp) pair per thread, and
// writes only the per-row logsumexp and loss; the backward reads them once
// more and writes the gradient directly in the dtype its consumer (the LM-head
// products) reads. Neither materialises log-probabilities or a one-hot.
//
// Rows of any length move 16 bytes at a time: row r starts at element r V, so up to 31
// elements at its head and three at its tail are taken alone, and what lies between starts
// at a 128-byte line of the logits (at a 16-byte boundary within a line the non-temporal
// stores of two waves share lines: backward of 4096 x 50257 372 us, from the line's start
// 317). us on one MI355X, before / now, forward and backward with a float gradient:
//   8192 x 32768 (1 GiB): 170 / 157 (6.8 TB/s) and 420 / 402 (5.3 TB/s, 92% of a copy's rate)
//   4096 x 50257: 254 / 123 and 382 / 317      500 x 131071: 179 / 48 and 293 / 96
//   16384 x 256: 16 / 7 and 8 / 6.5            8192 x 2048: 16 / 11 and 23 / 21.5
#include <math.h>

#include <algorithm>

#include "common.h"

namespace ferrite {
namespace {

constexpr int kCeThreads = 256;

// Merge two (max, sum of exp(x - max)) pairs.
__device__ __forceinline__ void ms_merge(float& m, float& s, float m2, float s2) {
  if (m2 == m) {  // also where both are infinite
    s += s2;
  } else if (m2 > m) {
    s = s * __expf(m - m2) + s2;
    m = m2;
  } else if (m2 > -INFINITY) {
    s += s2 * __expf(m2 - m);
  }
}

// Adds N elements to (m, s): one rescale for all of them. -inf adds nothing (nor does NaN), an
// element equal to the new max adds 1 (also where both are +inf).
template <int N>
__device__ __forceinline__ void ms_add(float& m, float& s, const float (&x)[N]) {
  float mn = m;
#pragma unroll
  for (int e = 0; e < N; ++e) mn = fmaxf(mn, x[e]);
  if (mn == -INFINITY) return;
  float t = m == mn ? s : s * __expf(m - mn);
#pragma unroll
  for (int e = 0; e < N; ++e) t += x[e] == mn ? 1.f : x[e] > -INFINITY ? __expf(x[e] - mn) : 0.f;
  m = mn;
  s = t;
}

constexpr int kLine = 32;  // floats in a 128-byte line

// How a row of V elements at element index row V splits: `head` elements alone, then `vecs`
// 16-byte vectors, then the tail from element `tail` on. VEC = false (an unaligned base): all tail.
struct RowSplit {
  int head;
  int64_t vecs, tail;
};
template <bool VEC>
__device__ __forceinline__ RowSplit split_row(int64_t row, int64_t V) {
  if (!VEC) return {0, 0, 0};
  const int head = (int)std::min<int64_t>((kLine - ((row * V) & (kLine - 1))) & (kLine - 1), V);
  const int64_t vecs = (V - head) / 4;
  return {head, vecs, head + 4 * vecs};
}

constexpr int kCeBatch = 4;  // vectors a thread loads together

// lse[row] = max + log(sum exp(x - max)), loss[row] = lse - x[target]. WPR waves per row: a
// workgroup of four for long rows, one wave for short ones, which then share a workgroup.
template <bool VEC, int WPR>
__global__ __launch_bounds__(kCeThreads) void ce_fwd_kernel(const float* __restrict__ logits,
                                                           const int64_t* __restrict__ targets,
                                                           float* __restrict__ loss, float* __restrict__ lse,
                                                           int64_t N, int64_t V) {
  constexpr int T = 64 * WPR;
  const int64_t row = (int64_t)blockIdx.x * (kCeThreads / T) + threadIdx.x / T;
  if (row >= N) return;  // whole waves; a four-wave row is a workgroup of its own
  const int t = threadIdx.x % T;
  const float* x = logits + row * V;
  const RowSplit sp = split_row<VEC>(row, V);
  float m = -INFINITY, s = 0.f;
  const f32x4* xv = reinterpret_cast<const f32x4*>(x + sp.head);
  int64_t i = t;
  for (; i + (kCeBatch - 1) * T < sp.vecs; i += kCeBatch * T) {
    f32x4 v[kCeBatch];
#pragma unroll
    for (int u = 0; u < kCeBatch; ++u) v[u] = __builtin_nontemporal_load(xv + i + u * T);
    float e[4 * kCeBatch];
#pragma unroll
    for (int u = 0; u < 4 * kCeBatch; ++u) e[u] = v[u / 4][u % 4];
    ms_add(m, s, e);
  }
  for (; i < sp.vecs; i += T) {
    const f32x4 v = __builtin_nontemporal_load(xv + i);
    const float e[4] = {v[0], v[1], v[2], v[3]};
    ms_add(m, s, e);
  }
  if (t < sp.head) {
    const float e[1] = {x[t]};
    ms_add(m, s, e);
  }
  for (int64_t k = sp.tail + t; k < V; k += T) {
    const float e[1] = {x[k]};
    ms_add(m, s, e);
  }
  // wave, then workgroup merge (fixed order)
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float m2 = __shfl_xor(m, off, kWave), s2 = __shfl_xor(s, off, kWave);
    ms_merge(m, s, m2, s2);
  }
  if constexpr (WPR > 1) {
    __shared__ float sm[WPR], ss[WPR];
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
      sm[wave] = m;
      ss[wave] = s;
    }
    __syncthreads();
    m = sm[0];
    s = ss[0];
    for (int w = 1; w < WPR; ++w) ms_merge(m, s, sm[w], ss[w]);
  }
  if (t == 0) {
    const float l = m + logf(s);
    lse[row] = l;
    const int64_t k = targets[row];
    loss[row] = (k >= 0 && k < V) ? l - x[k] : NAN;
  }
}

// grad[row, j] = (exp(x - lse[row]) - [j == target]) * (*dloss) * scale.
template <typename TO, bool VEC, int WPR>
__global__ __launch_bounds__(kCeThreads) void ce_bwd_kernel(const float* __restrict__ logits,
                                                           const int64_t* __restrict__ targets,
                                                           const float* __restrict__ lse,
                                                           const float* __restrict__ dloss, float scale,
                                                           TO* __restrict__ grad, int64_t N, int64_t V) {
  constexpr int T = 64 * WPR;
  const int64_t row = (int64_t)blockIdx.x * (kCeThreads / T) + threadIdx.x / T;
  if (row >= N) return;
  const int t = threadIdx.x % T;
  const float* x = logits + row * V;
  TO* gr = grad + row * V;
  const RowSplit sp = split_row<VEC>(row, V);
  const float l = lse[row];
  const float c = *dloss * scale;
  const int64_t k = targets[row];
  auto one = [&](float v, int64_t j) { return (__expf(v - l) - (j == k ? 1.f : 0.f)) * c; };
  const f32x4* xv = reinterpret_cast<const f32x4*>(x + sp.head);
  auto put = [&](const f32x4& v, int64_t i) {
    const int64_t j = sp.head + 4 * i;
    const float o[4] = {one(v[0], j), one(v[1], j + 1), one(v[2], j + 2), one(v[3], j + 3)};
    if constexpr (sizeof(TO) == 2)
      __builtin_nontemporal_store(bf16x4{(bf16)o[0], (bf16)o[1], (bf16)o[2], (bf16)o[3]}, reinterpret_cast<bf16x4*>(gr + j));
    else
      __builtin_nontemporal_store(f32x4{o[0], o[1], o[2], o[3]}, reinterpret_cast<f32x4*>(gr + j));
  };
  int64_t i = t;
  for (; i + (kCeBatch - 1) * T < sp.vecs; i += kCeBatch * T) {
    f32x4 v[kCeBatch];
#pragma unroll
    for (int u = 0; u < kCeBatch; ++u) v[u] = __builtin_nontemporal_load(xv + i + u * T);
#pragma unroll
    for (int u = 0; u < kCeBatch; ++u) put(v[u], i + u * T);
  }
  for (; i < sp.vecs; i += T) put(__builtin_nontemporal_load(xv + i), i);
  if (t < sp.head) gr[t] = Elem<TO>::from_f32(one(x[t], t));
  for (int64_t j = sp.tail + t; j < V; j += T) gr[j] = Elem<TO>::from_f32(one(x[j], j));
}

// Waves per row. Many short rows take one each, four to a workgroup: a workgroup's merge costs more than it
// saves (forward, four waves / one: 4096 x 2048 12.7 / 9.4 us, 16384 x 1000 30 / 20, 65536 x 512 91 / 37; up to
// 512 columns at any number of rows, 64 x 512 5.0 / 4.9), but few rows leave most CUs idle and wait
// for their chains (64 x 1000 5.1 / 6.4, 512 x 2000 6.0 / 8.6, 1024 x 700 5.5 / 6.3). The backward, which
// merges nothing, takes one up to 512 columns (16384 x 256 12.1 / 8.1) and two of many rows up to
// 1536 (four / two: 4096 x 700 8.1 / 7.4; 512 x 2000 4.9 / 6.6, 4096 x 2000 13.6 / 15.4).
constexpr int64_t kOneWave = 512, kManyRows = 2048;
bool one_wave_fwd(int64_t n, int64_t v) { return v <= kOneWave || (n > kManyRows && v <= 2048); }
bool two_waves_bwd(int64_t n, int64_t v) { return n > kManyRows && v <= 1536; }

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace ferrite

extern "C" int ferrite_hip_cross_entropy_fwd(const float* logits, const int64_t* targets, float* loss, float* lse,
                                             int64_t n, int64_t v, void* stream) {
  using namespace ferrite;
  if (n < 0 || v < 1) return fail(FERRITE_ERR_INVALID_ARGUMENT, "ferrite_hip_cross_entropy_fwd: need n >= 0, v >= 1");
  if (n > 0x7fffffff) return fail(FERRITE_ERR_INVALID_ARGUMENT, "ferrite_hip_cross_entropy_fwd: too many rows");
  if (n == 0) return FERRITE_OK;
  if (!logits || !targets || !loss || !lse)
    return fail(FERRITE_ERR_INVALID_ARGUMENT, "ferrite_hip_cross_entropy_fwd: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool vec = aligned16(logits);
  auto go = [&](auto kern, int per_block) {
    hipLaunchKernelGGL(kern, dim3((unsigned)cdiv(n, (int64_t)per_block)), dim3(kCeThreads), 0, s, logits, targets, loss,
                       lse, n, v);
  };
  if (one_wave_fwd(n, v))
    vec ? go(ce_fwd_kernel<true, 1>, 4) : go(ce_fwd_kernel<false, 1>, 4);
  else
    vec ? go(ce_fwd_kernel<true, 4>, 1) : go(ce_fwd_kernel<false, 4>, 1);
  return check_launch("ferrite_cross_entropy_fwd");
}

extern "C" int ferrite_hip_cross_entropy_bwd(const float* logits, const int64_t* targets, const float* lse,
                                             const float* dloss, float scale, void* grad, int64_t n, int64_t v,
                                             int grad_dtype, void* stream) {
  using namespace ferrite;
  if (!valid_dtype(grad_dtype))
    return fail(FERRITE_ERR_INVALID_ARGUMENT, "ferrite_hip_cross_entropy_bwd: dtype must be FERRITE_F32 or FERRITE_BF16");
  if (n < 0 || v < 1) return fail(FERRITE_ERR_INVALID_ARGUMENT, "ferrite_hip_cross_entropy_bwd: need n >= 0, v >= 1");
  if (n > 0x7fffffff) return fail(FERRITE_ERR_INVALID_ARGUMENT, "ferrite_hip_cross_entropy_bwd: too many rows");
  if (n == 0) return FERRITE_OK;
  if (!logits || !targets || !lse || !dloss || !grad)
    return fail(FERRITE_ERR_INVALID_ARGUMENT, "ferrite_hip_cross_entropy_bwd: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool vec = aligned16(logits) && aligned16(grad);
  auto go = [&](auto kern, int per_block, auto* g) {
    hipLaunchKernelGGL(kern, dim3((unsigned)cdiv(n, (int64_t)per_block)), dim3(kCeThreads), 0, s, logits, targets, lse,
                       dloss, scale, g, n, v);
  };
  auto rows = [&](auto* g) {
    typedef std::remove_pointer_t<decltype(g)> TO;
    if (v <= kOneWave)
      vec ? go(ce_bwd_kernel<TO, true, 1>, 4, g) : go(ce_bwd_kernel<TO, false, 1>, 4, g);
    else if (two_waves_bwd(n, v))
      vec ? go(ce_bwd_kernel<TO, true, 2>, 2, g) : go(ce_bwd_kernel<TO, false, 2>, 2, g);
    else
      vec ? go(ce_bwd_kernel<TO, true, 4>, 1, g) : go(ce_bwd_kernel<TO, false, 4>, 1, g);
  };
  if (grad_dtype == FERRITE_BF16)
    rows(static_cast<bf16*>(grad));
  else
    rows(static_cast<float*>(grad));
  return check_launch("ferrite_cross_entropy_bwd");
}
