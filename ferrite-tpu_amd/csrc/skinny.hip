// Products of few rows, out[M,N] = x[M,K] . w with M <= 64, for gfx950: a decode step's
// linear layers, and the input gradients of such layers.
//
// Reference: src/ferrite/kernels/matmul.py:27-38 (the blocked matmul, which pads a few rows
// to a block) and model/gpt.py:95-104 (the linear layer that rounds its weight to the
// activations' dtype).
//
// Bound by reading w once: M is at most two MFMA blocks of 32 rows, so a 256-row tile would
// spend its products on padding and leave one workgroup per 256 columns to read w. Here a
// workgroup owns 32 C columns and up to 16 waves share K between them, 16 k at a time in
// turn, so a workgroup keeps 16 waves' loads in flight and the whole K is read in a few
// round trips. The waves' f32 sums meet in LDS and are added in wave order (deterministic).
// What is left is the latency of those round trips: 8 x 512 . 512 x 2048 takes 4.3 us
// (11.8 before) where a launch alone takes about 3, 8 x 4096 . 4096 x 4096 13.5 us, 2.5 TB/s.
// No LDS stands between memory and the products: as A operand (w^T) a lane needs 8
// consecutive k of one column, and it gets them by loading 8 rows of its column and pairing
// them in registers, a v_perm (bf16) or a v_cvt_pk_bf16_f32 (float w) per pair; the 32
// lanes of a row read 32 C consecutive elements. Out of range rows and columns read as
// zeros through the descriptor's range.
#include "skinny.h"

#include <algorithm>

#include "gelu.h"
#include "splitk.h"

namespace ferrite {
namespace {

constexpr int kMaxWaves = 16;
constexpr uint32_t kOut = 0x80000000u;  // an offset past every descriptor's range

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* p, int64_t bytes) {
  const u32x4 r = buffer_rsrc(p, (uint32_t)(bytes < 0 ? 0 : bytes < 0x7ffffff0 ? bytes : 0x7ffffff0));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((uint64_t)r[1] << 32) | r[0]), (short)0, (int)r[2],
                                           0x00020000);
}
__device__ __forceinline__ uint32_t load_b16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0);
}

// The 8 elements of x row `row` from k0 + k (zeros past K and past M). `r` starts at column k0.
template <bool AL>
__device__ __forceinline__ u32x4 load_x(__amdgpu_buffer_rsrc_t r, uint32_t row_off, int k, int rem) {
  if constexpr (AL) {
    return __builtin_bit_cast(
        u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(k < rem ? row_off + 2 * k : kOut), 0, 0));
  } else {
    u32x4 v;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint32_t lo = load_b16(r, k + 2 * d < rem ? row_off + 2 * (k + 2 * d) : kOut);
      const uint32_t hi = load_b16(r, k + 2 * d + 1 < rem ? row_off + 2 * (k + 2 * d + 1) : kOut);
      v[d] = lo | (hi << 16);
    }
    return v;
  }
}

// Adds the waves' accumulators and stores the workgroup's columns n0 .. n0 + 32 C - 1.
// acc[e][b] holds C^T of columns n0 + C j + e (j = 0..31): register r of lane (l32, g) is row
// 32 b + l32, j = (r / 4) * 8 + 4 g + r % 4.
template <typename TO, int C, int MB, int EPI>
__device__ __forceinline__ void reduce_store(const f32x16 (&acc)[C][MB], float* red, TO* out, bf16* aux, int M, int N,
                                             int n0, int waves) {
  constexpr int kCols = 32 * C, kPitch = kCols + 1;  // an odd pitch: the 32 rows of a store on 32 banks
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5, wave = threadIdx.x >> 6;
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const int rows = min(M - 32 * b, 32);
    if (rows <= 0) break;
    if (b > 0) __syncthreads();
    if (l32 < rows) {
      float* const dst = red + (wave * rows + l32) * kPitch;
#pragma unroll
      for (int e = 0; e < C; ++e)
#pragma unroll
        for (int r = 0; r < 16; ++r) dst[((r >> 2) * 8 + 4 * g + (r & 3)) * C + e] = acc[e][b][r];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < rows * kCols; i += blockDim.x) {
      const int m = i / kCols, c = i % kCols, n = n0 + c;
      float v = 0.f;
      for (int w = 0; w < waves; ++w) v += red[(w * rows + m) * kPitch + c];
      if (n >= N) continue;
      const int64_t at = (int64_t)(32 * b + m) * N + n;
      if constexpr (EPI == kEpiNone) {
        out[at] = Elem<TO>::from_f32(v);
      } else if constexpr (EPI == kEpiGelu) {
        const bf16 u = (bf16)v;
        aux[at] = u;
        out[at] = (bf16)gelu_tanh((float)u);
      } else {
        out[at] = (bf16)((float)(bf16)v * gelu_tanh_grad((float)aux[at]));
      }
    }
  }
}

__device__ __forceinline__ int xcd_block() {  // neighbouring columns on one XCD's L2
  const int n = (int)gridDim.x, b = (int)blockIdx.x;
  return n % 8 == 0 ? (b % 8) * (n / 8) + b / 8 : b;
}

// w [K,N]. C columns per lane: 2 where rows hold whole pairs (N even, w aligned to a pair),
// else 1. U of a wave's steps of 16 k are loaded together.
template <typename TW, typename TO, int C, int MB, int EPI, bool AL>
__global__ __launch_bounds__(64 * kMaxWaves) void gemm_skinny_kernel(const bf16* __restrict__ x,
                                                                     const TW* __restrict__ w, TO* __restrict__ out,
                                                                     bf16* __restrict__ aux, int M, int N, int K,
                                                                     int kslice, int64_t slab) {
  extern __shared__ float red[];
  // 128 registers for each of 16 waves
  constexpr int U = C * MB == 1 && AL ? 4 : C * MB < 4 ? 2 : 1;
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int n0 = xcd_block() * 32 * C;
  const int sbeg = (int)blockIdx.y * (kslice / 16), steps = min((K + 15) / 16, sbeg + kslice / 16);
  out += blockIdx.y * slab;
  uint32_t woff[8], xoff[MB];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    woff[i] = n0 + l32 * C < N ? (uint32_t)(((8 * g + i) * (int64_t)N + l32 * C) * sizeof(TW)) : kOut;
#pragma unroll
  for (int b = 0; b < MB; ++b) xoff[b] = l32 + 32 * b < M ? (uint32_t)((int64_t)(l32 + 32 * b) * K * 2) : kOut;

  f32x16 acc[C][MB];
#pragma unroll
  for (int e = 0; e < C; ++e)
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[e][b][r] = 0.f;

  for (int s = sbeg + wave; s < steps; s += waves * U) {
    uint32_t raw[U][8][sizeof(TW) == 2 ? 1 : C];  // the row's C elements (bf16: in one word)
    u32x4 xr[U][MB];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k0 = (s + u * waves) * 16;
      const int rem = s + u * waves < steps ? K - k0 : 0;  // past the slice: an empty range, zeros
      const __amdgpu_buffer_rsrc_t wr = rsrc_of(w + (rem > 0 ? (int64_t)k0 * N : 0) + n0,
                                                ((int64_t)min(rem, 16) * N - n0) * (int64_t)sizeof(TW));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if constexpr (sizeof(TW) == 2 && C == 1) {
          raw[u][i][0] = load_b16(wr, woff[i]);
        } else if constexpr (sizeof(TW) * C == 4) {
          raw[u][i][0] = __builtin_amdgcn_raw_buffer_load_b32(wr, (int)woff[i], 0, 0);
        } else {
          const auto v = __builtin_amdgcn_raw_buffer_load_b64(wr, (int)woff[i], 0, 0);
          raw[u][i][0] = v[0];
          raw[u][i][1] = v[1];
        }
      }
      const __amdgpu_buffer_rsrc_t xrs = rsrc_of(x + (rem > 0 ? k0 : 0), rem > 0 ? ((int64_t)M * K - k0) * 2 : 0);
#pragma unroll
      for (int b = 0; b < MB; ++b) xr[u][b] = load_x<AL>(xrs, xoff[b], 8 * g, xoff[b] == kOut ? 0 : rem);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < C; ++e) {
        u32x4 f;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          if constexpr (sizeof(TW) == 4)
            f[d] = pack_bf16(__uint_as_float(raw[u][2 * d][e]), __uint_as_float(raw[u][2 * d + 1][e]));
          else if constexpr (C == 1)
            f[d] = raw[u][2 * d][0] | (raw[u][2 * d + 1][0] << 16);
          else  // byte picks: the low or the high halves of the two rows
            f[d] = __builtin_amdgcn_perm(raw[u][2 * d + 1][0], raw[u][2 * d][0], e ? 0x07060302u : 0x05040100u);
        }
#pragma unroll
        for (int b = 0; b < MB; ++b)
          mma32(__builtin_bit_cast(bf16x8, f), __builtin_bit_cast(bf16x8, xr[u][b]), acc[e][b]);
      }
  }
  reduce_store<TO, C, MB, EPI>(acc, red, out, aux, M, N, n0, waves);
}

// The 8 elements of a float w row from k0 + k, rounded to bf16.
template <bool AL>
__device__ __forceinline__ u32x4 load_f32w(__amdgpu_buffer_rsrc_t r, uint32_t row_off, int k, int rem) {
  f32x8 v;
  if constexpr (AL) {
    const uint32_t at = k < rem ? row_off + 4 * k : kOut;  // + 16 stays past the range
    const f32x4 a = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)at, 0, 0));
    const f32x4 b = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(at + 16), 0, 0));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = a[e];
      v[4 + e] = b[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      v[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)(k + e < rem ? row_off + 4 * (k + e) : kOut), 0, 0));
  }
  return u32x4{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
}

// w given transposed, [N,K]: a lane's 8 k lie together. 64 k per step in four products:
// product i takes chunk 4 g + i of the step's eight 8-k chunks from both operands, so that
// a lane's four loads cover 64 consecutive bytes of its row (128 of a float w's).
template <typename TW, typename TO, int MB, int EPI, bool AL>
__global__ __launch_bounds__(64 * kMaxWaves) void gemm_skinny_t_kernel(const bf16* __restrict__ x,
                                                                       const TW* __restrict__ w, TO* __restrict__ out,
                                                                       bf16* __restrict__ aux, int M, int N, int K,
                                                                       int kslice, int64_t slab) {
  extern __shared__ float red[];
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int n0 = xcd_block() * 32;
  const int sbeg = (int)blockIdx.y * (kslice / 64), steps = min((K + 63) / 64, sbeg + kslice / 64);
  out += blockIdx.y * slab;
  const bool in = n0 + l32 < N;
  const uint32_t woff = (uint32_t)((int64_t)l32 * K * sizeof(TW));
  uint32_t xoff[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) xoff[b] = l32 + 32 * b < M ? (uint32_t)((int64_t)(l32 + 32 * b) * K * 2) : kOut;
  f32x16 acc[1][MB];
#pragma unroll
  for (int b = 0; b < MB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][b][r] = 0.f;
  for (int s = sbeg + wave; s < steps; s += waves) {
    const int k0 = s * 64, rem = K - k0;
    const __amdgpu_buffer_rsrc_t wr = rsrc_of(w + (int64_t)n0 * K + k0, ((int64_t)min(N - n0, 32) * K - k0) * (int64_t)sizeof(TW));
    const __amdgpu_buffer_rsrc_t xrs = rsrc_of(x + k0, ((int64_t)M * K - k0) * 2);
    // The chunks loaded together: all, or fewer where a chunk takes eight element loads.
    constexpr int F = AL ? (sizeof(TW) == 4 ? 2 : 4) : MB == 1 && sizeof(TW) == 2 ? 2 : 1;
#pragma clang loop unroll(disable)
    for (int i0 = 0; i0 < 4; i0 += F) {
      u32x4 wv[F], xv[F][MB];
#pragma unroll
      for (int i = 0; i < F; ++i) {
        const int k = (4 * g + i0 + i) * 8;
        if constexpr (sizeof(TW) == 4)
          wv[i] = load_f32w<AL>(wr, woff, k, in ? rem : 0);
        else
          wv[i] = load_x<AL>(wr, woff, k, in ? rem : 0);
#pragma unroll
        for (int b = 0; b < MB; ++b) xv[i][b] = load_x<AL>(xrs, xoff[b], k, xoff[b] == kOut ? 0 : rem);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int b = 0; b < MB; ++b)
          mma32(__builtin_bit_cast(bf16x8, wv[i]), __builtin_bit_cast(bf16x8, xv[i][b]), acc[0][b]);
    }
  }
  reduce_store<TO, 1, MB, EPI>(acc, red, out, aux, M, N, n0, waves);
}

bool x_aligned(const SkinnyArgs& a) {
  auto a16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  return a.k % 8 == 0 && a16(a.x) && (!a.w_t || a16(a.w));
}

// How a product is cut: columns per lane, and K slices in blockIdx.y whose f32 partials a
// second pass adds.
//
// Slices pay once a wave would read its K in more round trips than the second pass costs
// (about 3 us): from K = 4096 on, or 2048 with a second row block, as many as give 256
// workgroups, each at least 512 deep, at most 8. Two columns per lane halve the x reads per
// column and read 128-byte rows of a bf16 w; with fewer workgroups they pay only with slices
// or where N is large. us on one MI355X, bf16 w [K,N], M = 8, as one slice of one column /
// this rule / the 256-row tiles that ran before:
//   512 x 2048 (K x N) 4.3 / 4.3 / 11.8    2048 x 512 6.3 / 6.3 / 14.7
//   4096 x 1024 12.1 / 8.3 / 16.7          4096 x 4096 20.3 / 13.5 / 20.4
//   8192 x 2048 36.1 / 13.8 / 23.0         8192 x 8192 39.7 / 35.0 / 37.9
struct SkinnyPlan {
  int cols, slices, kslice;
};
SkinnyPlan skinny_plan(const SkinnyArgs& a) {
  const int64_t esize = a.w_dtype == FERRITE_F32 ? 4 : 2;
  // (Two row blocks of element-wise x leave no registers for two columns.)
  const bool pairs = !a.w_t && a.n % 2 == 0 && (reinterpret_cast<uintptr_t>(a.w) & (2 * esize - 1)) == 0 &&
                     (a.m <= 32 || x_aligned(a));
  SkinnyPlan p{};
  p.cols = pairs && (a.k >= 4096 || a.n > (a.m > 32 ? 4096 : 8192)) ? 2 : 1;
  const int64_t step = a.w_t ? 64 : 16;
  int64_t s = 1;
  if (a.k >= 4096 || (a.m > 32 && a.k >= 2048))
    s = std::max<int64_t>(1, std::min<int64_t>({256 / cdiv(a.n, (int64_t)32 * p.cols), a.k / 512, (int64_t)8}));
  p.kslice = (int)(cdiv(cdiv(a.k, s), step) * step);
  p.slices = (int)cdiv(a.k, (int64_t)p.kslice);
  return p;
}
int64_t slab_floats(const SkinnyArgs& a) { return cdiv(a.m * a.n, (int64_t)4) * 4; }

template <typename Kern, typename TW, typename TO>
int go(Kern kern, const SkinnyArgs& a, const SkinnyPlan& p, hipStream_t stream, const TW*, TO* out) {
  // A wave per step of the slice, up to 16 and a power of two, at least 4 (which share the sums).
  const int kstep = a.w_t ? 64 : 16, cols = 32 * p.cols;
  int waves = 4;
  while (waves < kMaxWaves && waves * kstep < p.kslice) waves *= 2;
  const int lds = waves * (int)std::min<int64_t>(a.m, 32) * (cols + 1) * (int)sizeof(float);
  if (int rc = allow_lds((const void*)kern, lds > 64 * 1024 ? 160 * 1024 : 64 * 1024, stream, "ferrite_matmul")) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)cdiv(a.n, (int64_t)cols), (unsigned)p.slices), dim3(64 * waves), lds, stream,
                     static_cast<const bf16*>(a.x), static_cast<const TW*>(a.w), out, static_cast<bf16*>(a.aux),
                     (int)a.m, (int)a.n, (int)a.k, p.kslice, p.slices > 1 ? slab_floats(a) : 0);
  return check_launch("ferrite_matmul");
}

template <typename TW, typename TO, int EPI, int MB, bool AL>
int launch(const SkinnyArgs& a, const SkinnyPlan& p, TO* out, hipStream_t stream) {
  const TW* tw = nullptr;
  if constexpr (sizeof(TW) == 2 || EPI == kEpiNone)
    if (a.w_t) return go(gemm_skinny_t_kernel<TW, TO, MB, EPI, AL>, a, p, stream, tw, out);
  if constexpr (AL || MB == 1)
    if (p.cols == 2) return go(gemm_skinny_kernel<TW, TO, 2, MB, EPI, AL>, a, p, stream, tw, out);
  return go(gemm_skinny_kernel<TW, TO, 1, MB, EPI, AL>, a, p, stream, tw, out);
}

template <typename TW, typename TO, int EPI>
int launch_al(const SkinnyArgs& a, const SkinnyPlan& p, void* out, hipStream_t stream) {
  const bool al = x_aligned(a);
  TO* o = static_cast<TO*>(out);
  if (a.m <= 32) return al ? launch<TW, TO, EPI, 1, true>(a, p, o, stream) : launch<TW, TO, EPI, 1, false>(a, p, o, stream);
  return al ? launch<TW, TO, EPI, 2, true>(a, p, o, stream) : launch<TW, TO, EPI, 2, false>(a, p, o, stream);
}

template <typename TO, int EPI>
int sum_slices(const SkinnyArgs& a, const SkinnyPlan& p, hipStream_t stream) {
  const int64_t mn = a.m * a.n;
  hipLaunchKernelGGL((gemm_splitk_reduce_kernel<TO, EPI>), dim3((unsigned)cdiv(mn, (int64_t)1024)), dim3(256), 0, stream,
                     static_cast<const float*>(a.ws), static_cast<TO*>(a.out), mn, p.slices, static_cast<bf16*>(a.aux),
                     slab_floats(a));
  return check_launch("ferrite_matmul");
}

template <typename TW>
int dispatch(const SkinnyArgs& a, hipStream_t stream) {
  SkinnyPlan p = skinny_plan(a);
  // The sum of the slabs leaves in 8-byte stores, and its GELU needs whole fours.
  if (!a.ws || a.ws_bytes < p.slices * slab_floats(a) * (int64_t)sizeof(float) ||
      (reinterpret_cast<uintptr_t>(a.ws) & 15) || (reinterpret_cast<uintptr_t>(a.out) & 7) ||
      (a.epi != kEpiNone && (a.m * a.n % 4 != 0 || (reinterpret_cast<uintptr_t>(a.aux) & 7)))) {
    p.slices = 1;
    p.kslice = (int)(cdiv(a.k, (int64_t)64) * 64);
  }
  if (p.slices > 1) {
    if (int rc = launch_al<TW, float, kEpiNone>(a, p, a.ws, stream)) return rc;
    if (a.epi == kEpiGelu) return sum_slices<bf16, kEpiGelu>(a, p, stream);
    if (a.epi == kEpiGeluGrad) return sum_slices<bf16, kEpiGeluGrad>(a, p, stream);
    return a.out_dtype == FERRITE_BF16 ? sum_slices<bf16, kEpiNone>(a, p, stream) : sum_slices<float, kEpiNone>(a, p, stream);
  }
  if (a.epi == kEpiGelu) return launch_al<TW, bf16, kEpiGelu>(a, p, a.out, stream);
  if constexpr (sizeof(TW) == 2)
    if (a.epi == kEpiGeluGrad) return launch_al<TW, bf16, kEpiGeluGrad>(a, p, a.out, stream);
  return a.out_dtype == FERRITE_BF16 ? launch_al<TW, bf16, kEpiNone>(a, p, a.out, stream)
                                     : launch_al<TW, float, kEpiNone>(a, p, a.out, stream);
}

}  // namespace

bool skinny_ok(int64_t m, int64_t n, int64_t k) {
  // 32-bit offsets within 64 rows of x and w^T and 16 rows of w; the grid.
  return m >= 1 && m <= kSkinnyRows && n <= 0x7fffffff / 64 && k <= 0x7fffffff / 128;
}

bool skinny_better(int64_t m, int64_t n, int64_t k) {
  return skinny_ok(m, n, k) && (n * k <= (int64_t)1 << 24 || (m <= 8 && k >= 4096));
}

int64_t skinny_workspace(const SkinnyArgs& a) {
  const SkinnyPlan p = skinny_plan(a);
  return p.slices > 1 ? p.slices * slab_floats(a) * (int64_t)sizeof(float) : 0;
}

int skinny_launch(const SkinnyArgs& a, hipStream_t stream) {
  return a.w_dtype == FERRITE_F32 ? dispatch<float>(a, stream) : dispatch<bf16>(a, stream);
}

}  // namespace ferrite
