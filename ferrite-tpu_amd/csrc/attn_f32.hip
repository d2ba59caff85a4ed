// Float32 attention for gfx950: forward, dQ and dK/dV for head dims up to 128.
//
// Reference: src/ferrite/kernels/flash_attention.py:91-175 (forward), :224-243 (dQ),
// :197-221 (dK/dV), at Precision.HIGHEST for f32 operands (_compat.py:17-25).
//
// Bound by the fp32 matrix rate: v_mfma_f32_32x32x2_f32 takes 64 cycles, so a 32 x 32 tile at
// head dim 64 keeps a SIMD's matrix pipe busy for 2048 cycles per product while it moves 8 KB.
// A wave's chain of tiles is therefore what lasts, and what has to be cut: a workgroup owns 32
// rows (queries; keys in dK/dV) and its four waves share the tiles of the other side between
// them, every fourth each, with a softmax state or gradient of their own that is combined
// through LDS at the end, in wave order (deterministic). With 128 rows per workgroup and whole
// sweeps per wave, 2x8x1024x64 was 128 workgroups on 256 CUs with sweeps of up to 32 tiles.
//
// At that rate operands need no LDS either: a wave loads its fragments straight from memory
// (the four waves' tiles come out of L2), row fragments as 16-byte loads of a lane's row, the
// transposed ones as 4-byte loads of a lane's column, each a stage ahead of its products, in
// registers that the stage before has just finished with. There is no barrier in the loop.
//
// Rows past the end read as zeros through the descriptor's range, columns past d through an
// offset outside it.
//
// us on one MI355X, 128 rows a workgroup / these, forward, dQ, dK/dV (flops of the causal half):
//   2x8x1024x64 causal   82 / 34 (63 TFLOP/s)    119 / 50    155 / 62
//   1x1x8192x64 causal   608 / 155               904 / 223   1197 / 327
//   1x8x4096x64 causal   308 / 158 (109)         459 / 235   606 / 356
//   5x1x128x80 causal    21 / 9.7                30 / 13     41 / 16
// The forward and dQ run two waves per SIMD up to head dim 64 (dQ of 4x16x1024x64 166 us with
// one, 133 with two); dK/dV's accumulators leave room for one (with two, 160 bytes spilled:
// 62 -> 94 us).
#include "attn_f32.h"

#include <math.h>

#include <algorithm>

namespace ferrite {
namespace {

constexpr int kWaves = 4;
constexpr uint32_t kOut = 0x80000000u;
constexpr float kRescale = 8.f;  // log2: the running max may lag a row's true one by this much

// Row of the tile that accumulator row order gives lane row p: S^T = K Q^T computed over rows taken
// in this order has its register r of lane group g at row 16 g + r of the tile.
__device__ __forceinline__ int row_of_lane(int p) {
  return (((p >> 2) & 1) << 4) | (((p >> 4) & 1) << 3) | (((p >> 3) & 1) << 2) | (p & 3);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_from(const float* base, int row0, int nrows, int d) {
  const u32x4 r = buffer_rsrc(base + (int64_t)row0 * d, (uint32_t)(max(nrows - row0, 0) * d * 4));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((uint64_t)r[1] << 32) | r[0]), (short)0, (int)r[2],
                                           0x00020000);
}

// Fragments of rows: lane (l32, g) takes elements 16 kk + 8 g .. + 7 of row `row` past the base.
// FULL: d == D, so that the offsets differ by constants alone.
template <int D, bool FULL>
__device__ __forceinline__ void load_rows(f32x8 (&f)[D / 16], __amdgpu_buffer_rsrc_t r, int row, int g, int d) {
  const uint32_t row_at = (uint32_t)((row * d + 8 * g) * 4);
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    const int c = 16 * kk + 8 * g;
    const uint32_t at = row_at + 64 * kk;
    const f32x4 a =
        __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(FULL || c < d ? at : kOut), 0, 0));
    const f32x4 b = __builtin_bit_cast(
        f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(FULL || c + 4 < d ? at + 16 : kOut), 0, 0));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[kk][e] = a[e];
      f[kk][4 + e] = b[e];
    }
  }
}

// Fragments of the transposed tile of rows row0 ..: f[u][h] of lane (l32, g) is column 32 u + l32 of
// rows 16 g + 8 h .. + 7. Each of the 16 row steps is a descriptor of its own, formed on the scalar
// unit: 16 D / 32 lane offsets would not fit beside the accumulators.
template <int D, bool FULL>
__device__ __forceinline__ void load_cols(f32x8 (&f)[D / 32][2], const float* base, int row0, int nrows, int l32, int g,
                                          int d) {
  const uint32_t at = (uint32_t)((16 * g * d + l32) * 4);
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const __amdgpu_buffer_rsrc_t r = rows_from(base, row0 + 8 * h + e, nrows, d);
#pragma unroll
      for (int u = 0; u < D / 32; ++u)
        f[u][h][e] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)(FULL || 32 * u + l32 < d ? at + 128 * u : kOut), 0, 0));
    }
}

template <int N>
__device__ __forceinline__ void clear(f32x16 (&a)[N]) {
#pragma unroll
  for (int u = 0; u < N; ++u)
#pragma unroll
    for (int r = 0; r < 16; ++r) a[u][r] = 0.f;
}
template <int D>
__device__ __forceinline__ f32x16 dot_rows(const f32x8 (&a)[D / 16], const f32x8 (&b)[D / 16]) {
  f32x16 s;
#pragma unroll
  for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) mma32(a[kk], b[kk], s);
  return s;
}
// acc (D x 32) += cols^T (D x 32 rows) . p (32 rows x 32), p as dot_rows leaves it.
template <int D>
__device__ __forceinline__ void add_cols(const f32x8 (&cols)[D / 32][2], const f32x16& p, f32x16 (&acc)[D / 32]) {
  f32x8 b[2];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    b[0][e] = p[e];
    b[1][e] = p[8 + e];
  }
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int e = 0; e < 8; ++e)  // consecutive products on different accumulators
#pragma unroll
      for (int u = 0; u < D / 32; ++u)
        acc[u] = __builtin_amdgcn_mfma_f32_32x32x2f32(cols[u][h][e], b[h][e], acc[u], 0, 0, 0);
}

// The sum over the waves of acc (D x 32, a column per output row) times mul, stored as the rows
// `row` = row0 + l32 of out: each wave leaves its registers in LDS, then adds D / 32 quads of them
// in wave order. Call it by whole workgroups; it ends with its LDS free for the next call.
template <int D>
__device__ __forceinline__ void sum_store(const f32x16 (&acc)[D / 32], float* lds, float* out, int row, int nrows, int d,
                                          float mul) {
  const int lane = threadIdx.x & 63, g = lane >> 5, wave = threadIdx.x >> 6;
  constexpr int kRegs = D / 2;  // accumulator registers of a wave
#pragma unroll
  for (int u = 0; u < D / 32; ++u)
#pragma unroll
    for (int r = 0; r < 16; ++r) lds[(wave * kRegs + u * 16 + r) * 64 + lane] = acc[u][r];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < D / 32; ++i) {
    const int quad = wave * (D / 32) + i, c = (quad >> 2) * 32 + (quad & 3) * 8 + g * 4;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += lds[(w * kRegs + quad * 4 + e) * 64 + lane];
    if (row < nrows && c < d) *reinterpret_cast<f32x4*>(out + (int64_t)row * d + c) = v * mul;  // d % 4 == 0
  }
  __syncthreads();
}

template <int D, bool FULL>
__global__ __launch_bounds__(64 * kWaves, D <= 64 ? 2 : 1) void attn_fwd_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, float* __restrict__ o,
    float* __restrict__ lse, int bh_count, int Sq, int Sk, int d, int causal, float scale_log2, float q_sign, int n_qtiles) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ float ml[2][kWaves][32];
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Heaviest (last) query tiles first; the tiles of one head share an XCD when bh_count % 8 == 0.
  const int bh = blockIdx.x % bh_count, q0 = (n_qtiles - 1 - (int)(blockIdx.x / bh_count)) * 32;
  const int qrow = q0 + l32;
  q += (int64_t)bh * Sq * d;
  k += (int64_t)bh * Sk * d;
  v += (int64_t)bh * Sk * d;
  const int n_tiles = causal ? min(min(q0 + 31, Sq - 1), Sk - 1) / 32 + 1 : (Sk + 31) / 32;
  f32x8 qf[D / 16], kf[D / 16], vf[D / 32][2];
  load_rows<D, FULL>(qf, rows_from(q, q0, Sq, d), l32, g, d);
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) qf[kk] *= q_sign;
  const int krow = row_of_lane(l32);
  load_rows<D, FULL>(kf, rows_from(k, wave * 32, Sk, d), krow, g, d);
  f32x16 acc[D / 32];
  clear(acc);
  float m = -INFINITY, lsum[4] = {0.f, 0.f, 0.f, 0.f};
  for (int j = wave; j < n_tiles; j += kWaves) {
    const int kv0 = j * 32;
    load_cols<D, FULL>(vf, v, kv0, Sk, l32, g, d);
    __builtin_amdgcn_sched_barrier(0);
    f32x16 s = dot_rows<D>(kf, qf);  // s[r]: key kv0 + 16 g + r, query qrow
    __builtin_amdgcn_sched_barrier(0);
    load_rows<D, FULL>(kf, rows_from(k, min(kv0 + 32 * kWaves, Sk), Sk, d), krow, g, d);  // past the end: nothing
    __builtin_amdgcn_sched_barrier(0);
    if ((causal && kv0 + 31 > q0) || kv0 + 32 > Sk) {
      const int lim = causal ? min(qrow, Sk - 1) : Sk - 1;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = kv0 + 16 * g + r > lim ? -INFINITY : s[r];
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = lane32_max(mx) * scale_log2;
    if (__any(mx > m + kRescale)) {
      const float m_new = fmaxf(m, mx);
      const float alpha = m_new > -INFINITY ? __builtin_amdgcn_exp2f(m - m_new) : 1.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) lsum[i] *= alpha;
#pragma unroll
      for (int u = 0; u < D / 32; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[u][r] *= alpha;
      m = m_new;
    }
    const float neg_m = m > -INFINITY ? -m : 0.f;  // a row with no key in this wave's tiles so far
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], scale_log2, neg_m));
      lsum[r & 3] += s[r];
    }
    add_cols<D>(vf, s, acc);
  }
  const float l = lane32_sum((lsum[0] + lsum[1]) + (lsum[2] + lsum[3]));
  if (g == 0) {
    ml[0][wave][l32] = m;
    ml[1][wave][l32] = l;
  }
  __syncthreads();
  float mt = ml[0][0][l32], lt = 0.f;
#pragma unroll
  for (int w = 1; w < kWaves; ++w) mt = fmaxf(mt, ml[0][w][l32]);
  auto weight = [&](float mw) { return mw > -INFINITY ? __builtin_amdgcn_exp2f(mw - mt) : 0.f; };
#pragma unroll
  for (int w = 0; w < kWaves; ++w) lt += ml[1][w][l32] * weight(ml[0][w][l32]);
  const float f = weight(m);
#pragma unroll
  for (int u = 0; u < D / 32; ++u)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[u][r] *= f;
  sum_store<D>(acc, lds, o + (int64_t)bh * Sq * d, qrow, Sq, d, 1.0f / lt);
  if (wave == 0 && g == 0 && qrow < Sq) lse[(int64_t)bh * Sq + qrow] = (mt + __builtin_amdgcn_logf(lt)) * kLn2;
}

template <int D, bool FULL>
__global__ __launch_bounds__(64 * kWaves, D <= 64 ? 2 : 1) void attn_dq_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ dout, const float* __restrict__ lse, const float* __restrict__ delta,
    float* __restrict__ dq, int bh_count, int Sq, int Sk, int d, int causal, float scale, int n_qtiles) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int bh = blockIdx.x % bh_count, q0 = (n_qtiles - 1 - (int)(blockIdx.x / bh_count)) * 32;
  const int qrow = q0 + l32;
  q += (int64_t)bh * Sq * d;
  dout += (int64_t)bh * Sq * d;
  k += (int64_t)bh * Sk * d;
  v += (int64_t)bh * Sk * d;
  const int n_tiles = causal ? min(min(q0 + 31, Sq - 1), Sk - 1) / 32 + 1 : (Sk + 31) / 32;
  const float scale_log2 = scale * kLog2e;
  f32x8 qf[D / 16], of[D / 16], kf[D / 16], vf[D / 16], kc[D / 32][2];
  load_rows<D, FULL>(qf, rows_from(q, q0, Sq, d), l32, g, d);
  load_rows<D, FULL>(of, rows_from(dout, q0, Sq, d), l32, g, d);
  const float nlse = qrow < Sq ? -lse[(int64_t)bh * Sq + qrow] * kLog2e : 0.f;
  const float dl = qrow < Sq ? delta[(int64_t)bh * Sq + qrow] : 0.f;
  const int krow = row_of_lane(l32);
  load_rows<D, FULL>(kf, rows_from(k, wave * 32, Sk, d), krow, g, d);
  load_rows<D, FULL>(vf, rows_from(v, wave * 32, Sk, d), krow, g, d);
  f32x16 acc[D / 32];
  clear(acc);
  for (int j = wave; j < n_tiles; j += kWaves) {
    const int kv0 = j * 32, next = min(kv0 + 32 * kWaves, Sk);
    load_cols<D, FULL>(kc, k, kv0, Sk, l32, g, d);
    __builtin_amdgcn_sched_barrier(0);
    f32x16 s = dot_rows<D>(kf, qf);
    __builtin_amdgcn_sched_barrier(0);
    load_rows<D, FULL>(kf, rows_from(k, next, Sk, d), krow, g, d);
    __builtin_amdgcn_sched_barrier(0);
    const f32x16 dp = dot_rows<D>(vf, of);
    __builtin_amdgcn_sched_barrier(0);
    load_rows<D, FULL>(vf, rows_from(v, next, Sk, d), krow, g, d);
    __builtin_amdgcn_sched_barrier(0);
    const bool edge = (causal && kv0 + 31 > q0) || kv0 + 32 > Sk;
    const int lim = causal ? min(qrow, Sk - 1) : Sk - 1;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], scale_log2, nlse));
      s[r] = edge && kv0 + 16 * g + r > lim ? 0.f : p * (dp[r] - dl) * scale;
    }
    add_cols<D>(kc, s, acc);
  }
  sum_store<D>(acc, lds, dq + (int64_t)bh * Sq * d, qrow, Sq, d, 1.f);
}

template <int D, bool FULL>
__global__ __launch_bounds__(64 * kWaves, 1) void attn_dkv_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ dout, const float* __restrict__ lse, const float* __restrict__ delta,
    float* __restrict__ dk, float* __restrict__ dv, int bh_count, int Sq, int Sk, int d, int causal, float scale) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // The first key tiles have the longest causal sweeps and come first.
  const int bh = blockIdx.x % bh_count, k0 = (int)(blockIdx.x / bh_count) * 32;
  const int krow = k0 + l32;
  q += (int64_t)bh * Sq * d;
  dout += (int64_t)bh * Sq * d;
  k += (int64_t)bh * Sk * d;
  v += (int64_t)bh * Sk * d;
  lse += (int64_t)bh * Sq;
  delta += (int64_t)bh * Sq;
  const int n_tiles = (Sq + 31) / 32;
  const float scale_log2 = scale * kLog2e;
  f32x8 kf[D / 16], vf[D / 16], qr[D / 16], orow[D / 16], qc[D / 32][2], oc[D / 32][2];
  load_rows<D, FULL>(kf, rows_from(k, k0, Sk, d), l32, g, d);
  load_rows<D, FULL>(vf, rows_from(v, k0, Sk, d), l32, g, d);
  f32x16 adk[D / 32], adv[D / 32];
  clear(adk);
  clear(adv);
  const int first = (causal ? k0 / 32 : 0) + wave, row = row_of_lane(l32);
  load_rows<D, FULL>(qr, rows_from(q, min(first * 32, Sq), Sq, d), row, g, d);
  for (int j = first; j < n_tiles; j += kWaves) {
    const int q0 = j * 32;
    load_rows<D, FULL>(orow, rows_from(dout, q0, Sq, d), row, g, d);
    // Statistics of the lane group's 16 queries (zeros past the end).
    f32x16 nl, dl;
    const __amdgpu_buffer_rsrc_t lr = rows_from(lse, q0, Sq, 1), dr = rows_from(delta, q0, Sq, 1);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      nl[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(lr, (16 * g + i) * 4, 0, 0));
      dl[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(dr, (16 * g + i) * 4, 0, 0));
    }
    __builtin_amdgcn_sched_barrier(0);
    f32x16 p = dot_rows<D>(qr, kf);  // p[r]: query q0 + 16 g + r, key krow
    __builtin_amdgcn_sched_barrier(0);
    load_cols<D, FULL>(oc, dout, q0, Sq, l32, g, d);
    __builtin_amdgcn_sched_barrier(0);
    f32x16 ds = dot_rows<D>(orow, vf);
    __builtin_amdgcn_sched_barrier(0);
    load_cols<D, FULL>(qc, q, q0, Sq, l32, g, d);
    __builtin_amdgcn_sched_barrier(0);
    const bool edge = causal && q0 < k0 + 31;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(p[r], scale_log2, -nl[r] * kLog2e));
      p[r] = edge && q0 + 16 * g + r < krow ? 0.f : pr;
      ds[r] = p[r] * (ds[r] - dl[r]) * scale;
    }
    add_cols<D>(oc, p, adv);
    __builtin_amdgcn_sched_barrier(0);
    load_rows<D, FULL>(qr, rows_from(q, min(q0 + 32 * kWaves, Sq), Sq, d), row, g, d);
    __builtin_amdgcn_sched_barrier(0);
    add_cols<D>(qc, ds, adk);
  }
  sum_store<D>(adk, lds, dk + (int64_t)bh * Sk * d, krow, Sk, d, 1.f);
  sum_store<D>(adv, lds, dv + (int64_t)bh * Sk * d, krow, Sk, d, 1.f);
}

template <int D>
constexpr int kLds = kWaves * (D / 2) * 64 * 4;

template <typename Kern, typename... Args>
int go(const char* what, Kern kern, int lds, int64_t tiles, int64_t bh, hipStream_t stream, Args... args) {
  if (tiles * bh > 0x7fffffff) return fail(FERRITE_ERR_INVALID_ARGUMENT, std::string(what) + ": grid too large");
  if (int rc = allow_lds((const void*)kern, lds, stream, "ferrite_hip_attn")) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(tiles * bh)), dim3(64 * kWaves), lds, stream, args...);
  return check_launch(what);
}

}  // namespace

// pick(D) with the head dim's padded size as a constant.
#define FERRITE_F32_DIM(d, CALL)      \
  do {                                \
    if ((d) <= 32) return CALL(32);   \
    if ((d) <= 64) return CALL(64);   \
    return CALL(128);                 \
  } while (0)

int f32_attn_fwd(const float* q, const float* k, const float* v, float* o, float* lse, const F32Attn& s, float scale,
                 hipStream_t stream) {
  // The row max is taken on raw scores, which needs a positive multiplier: a negative scale
  // negates q instead, and a zero scale becomes a tiny positive one (uniform weights either way).
  float c = scale * kLog2e;
  const float sign = c < 0.f ? -1.f : 1.f;
  c = fmaxf(fabsf(c), 1e-30f);
  const int64_t nq = cdiv(s.sq, (int64_t)32);
#define FERRITE_FWD(D)                                                                                             \
  go("ferrite_flash_attention_fwd", (s.d == D ? attn_fwd_f32_kernel<D, true> : attn_fwd_f32_kernel<D, false>), kLds<D>, nq, s.bh, stream, q, k, v, o, lse, (int)s.bh, \
     (int)s.sq, (int)s.sk, (int)s.d, s.causal, c, sign, (int)nq)
  FERRITE_F32_DIM(s.d, FERRITE_FWD);
#undef FERRITE_FWD
}

int f32_attn_dq(const float* q, const float* k, const float* v, const float* dout, const float* lse, const float* delta,
                float* dq, const F32Attn& s, float scale, hipStream_t stream) {
  const int64_t nq = cdiv(s.sq, (int64_t)32);
#define FERRITE_DQ(D)                                                                                              \
  go("ferrite_flash_attention_bwd_dq", (s.d == D ? attn_dq_f32_kernel<D, true> : attn_dq_f32_kernel<D, false>), kLds<D>, nq, s.bh, stream, q, k, v, dout, lse, delta, \
     dq, (int)s.bh, (int)s.sq, (int)s.sk, (int)s.d, s.causal, scale, (int)nq)
  FERRITE_F32_DIM(s.d, FERRITE_DQ);
#undef FERRITE_DQ
}

int f32_attn_dkv(const float* q, const float* k, const float* v, const float* dout, const float* lse,
                 const float* delta, float* dk, float* dv, const F32Attn& s, float scale, hipStream_t stream) {
  const int64_t nk = cdiv(s.sk, (int64_t)32);
#define FERRITE_DKV(D)                                                                                               \
  go("ferrite_flash_attention_bwd_dkv", (s.d == D ? attn_dkv_f32_kernel<D, true> : attn_dkv_f32_kernel<D, false>), kLds<D>, nk, s.bh, stream, q, k, v, dout, lse, delta, \
     dk, dv, (int)s.bh, (int)s.sq, (int)s.sk, (int)s.d, s.causal, scale)
  FERRITE_F32_DIM(s.d, FERRITE_DKV);
#undef FERRITE_DKV
}

}  // namespace ferrite
