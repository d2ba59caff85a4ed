// Head layout changes around the attention kernels, for gfx950.
//
// The QKV projection produces rows [G, H, D] per token ([B, S, G, H, D], G = 3
// for q, k, v), and the attention kernels read and write head-major
// [B, H, S, D] tensors; the attention output goes back to token-major rows
// ([B, S, H, D], G = 1) for the output projection. Reference: the transposes of
// src/ferrite/model/gpt.py:137-138, which XLA turns into copy fusions.
//
// HBM-bound permutes: every thread moves one 16-byte vector; the token-major
// side is read or written in whole contiguous rows and the head-major side in
// D-element runs, so both sides are coalesced.
#include <algorithm>

#include "common.h"
#include "internal_api.h"
#include "splitk.h"

namespace ferrite {
namespace {

constexpr int kMaxGroups = 4;

struct HeadPtrs {
  void* p[kMaxGroups];
};

// Element (b, s, g, h, e) of the token-major tensor <-> element (b, h, s, e) of
// head-major tensor g. V elements per thread (V = 16 bytes / sizeof(T), or 1).
template <typename T, int V, bool SPLIT>
__global__ __launch_bounds__(256) void heads_kernel(T* __restrict__ tok, HeadPtrs heads, int64_t S, int G, int H,
                                                    int D, int64_t total_vecs) {
  typedef __attribute__((ext_vector_type(4))) uint32_t vec_t;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total_vecs) return;
  const int dv = D / V;
  const int64_t row_vecs = (int64_t)G * H * dv;
  const int64_t bs = i / row_vecs;
  const int64_t c = i - bs * row_vecs;
  const int g = (int)(c / ((int64_t)H * dv));
  const int rem = (int)(c - (int64_t)g * H * dv);
  const int h = rem / dv, e = (rem - h * dv) * V;
  const int64_t b = bs / S, s = bs - b * S;
  T* head = static_cast<T*>(heads.p[g]) + ((b * H + h) * S + s) * D + e;
  T* t = tok + i * V;
  if constexpr (V * sizeof(T) == 16) {
    if constexpr (SPLIT)
      *reinterpret_cast<vec_t*>(head) = *reinterpret_cast<const vec_t*>(t);
    else
      *reinterpret_cast<vec_t*>(t) = *reinterpret_cast<const vec_t*>(head);
  } else {
    if constexpr (SPLIT)
      *head = *t;
    else
      *t = *head;
  }
}

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <typename T, bool SPLIT>
int heads_launch(void* tok, void* const* heads, int64_t B, int64_t S, int64_t G, int64_t H, int64_t D,
                 hipStream_t stream) {
  constexpr int kVec = 16 / sizeof(T);
  HeadPtrs hp{};
  bool vec = D % kVec == 0 && al16(tok);
  for (int g = 0; g < G; ++g) {
    hp.p[g] = heads[g];
    vec = vec && al16(heads[g]);
  }
  const int64_t elems = B * S * G * H * D;
  const int64_t total = vec ? elems / kVec : elems;
  const int64_t blocks = cdiv(total, 256);
  if (blocks > 0x7fffffff) return fail(FERRITE_ERR_INVALID_ARGUMENT, "ferrite_hip_heads: tensor too large");
  T* tp = static_cast<T*>(tok);
  if (vec)
    hipLaunchKernelGGL((heads_kernel<T, kVec, SPLIT>), dim3((unsigned)blocks), dim3(256), 0, stream, tp, hp, S, (int)G,
                       (int)H, (int)D, total);
  else
    hipLaunchKernelGGL((heads_kernel<T, 1, SPLIT>), dim3((unsigned)blocks), dim3(256), 0, stream, tp, hp, S, (int)G,
                       (int)H, (int)D, total);
  return check_launch(SPLIT ? "ferrite_heads_split" : "ferrite_heads_merge");
}

template <bool SPLIT>
int heads_dispatch(const char* name, void* tok, void* const* heads, int64_t b, int64_t s, int64_t g, int64_t h,
                   int64_t d, int dtype, void* stream) {
  if (!valid_dtype(dtype)) return fail(FERRITE_ERR_INVALID_ARGUMENT, std::string(name) + ": dtype must be FERRITE_F32 or FERRITE_BF16");
  if (b < 0 || s < 0 || g < 1 || g > kMaxGroups || h < 1 || d < 1 || g * h * d > 0x7fffffff)
    return fail(FERRITE_ERR_INVALID_ARGUMENT, std::string(name) + ": need b, s >= 0, 1 <= groups <= 4, heads, dim >= 1");
  if (b * s == 0) return FERRITE_OK;
  if (!tok || !heads) return fail(FERRITE_ERR_INVALID_ARGUMENT, std::string(name) + ": null pointer");
  for (int i = 0; i < g; ++i)
    if (!heads[i]) return fail(FERRITE_ERR_INVALID_ARGUMENT, std::string(name) + ": null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == FERRITE_BF16) return heads_launch<bf16, SPLIT>(tok, heads, b, s, g, h, d, st);
  return heads_launch<float, SPLIT>(tok, heads, b, s, g, h, d, st);
}

// The embedding, one block per row: of a decode step, where four launches of a tensor library (two
// gathers, the sum, the conversion) cost more than the rest of a short step's layer, and of a
// training step, where they move 130 bytes for 17 (16384 x 512, float tables). Without pos, row
// r is at position r % period. V elements per thread and pass: 4 of aligned rows, else 1.
template <typename TE, typename TO, int V>
__global__ __launch_bounds__(256) void embed_kernel(const int64_t* __restrict__ tokens, const int32_t* __restrict__ pos,
                                                    const TE* __restrict__ tok_emb, const TE* __restrict__ pos_emb,
                                                    TO* __restrict__ out, int64_t dim, int64_t vocab, int64_t seq,
                                                    int period) {
  typedef TE __attribute__((ext_vector_type(V))) in_t;
  typedef TO __attribute__((ext_vector_type(V))) out_t;
  const int64_t r = blockIdx.x;
  int64_t t = tokens[r], p = pos ? pos[r] : (int)blockIdx.x % period;
  t += t < 0 ? vocab : 0;
  p += p < 0 ? seq : 0;
  if (t < 0 || t >= vocab || p < 0 || p >= seq) __builtin_trap();
  for (int64_t e = (int64_t)threadIdx.x * V; e < dim; e += 256 * V) {
    const in_t a = *reinterpret_cast<const in_t*>(tok_emb + t * dim + e);
    const in_t b = *reinterpret_cast<const in_t*>(pos_emb + p * dim + e);
    out_t o;
#pragma unroll
    for (int i = 0; i < V; ++i)
      o[i] = Elem<TO>::from_f32(
          Elem<TE>::to_f32(Elem<TE>::from_f32(Elem<TE>::to_f32(a[i]) + Elem<TE>::to_f32(b[i]))));
    *reinterpret_cast<out_t*>(out + r * dim + e) = o;
  }
}

// The token table's gradient of a small vocabulary: rows of dh summed by token. A tensor library
// sorts the tokens and adds the many rows of each token one after another. Here a wave owns C
// columns (a lane each) of a slice of the rows and adds every row into its own [vocab, C] table
// in LDS, so nothing is sorted; a lane adds to its own column in row order and the slices' tables
// are summed in slice order (deterministic). C is what a 64 KB table leaves (two workgroups per
// CU): 64 up to 256 tokens, 32 up to 512 and 16 up to 1024, where the wave's 64 lanes load each dh
// element two and four times. Bound by the chain of table updates in a wave: LDS atomics took 59 us
// for 16384 x 512 bf16 over 256 tokens, reads and writes of two rows at a time 34; the sum of the
// 64 slices' tables takes 17.7 more and the position table 4.8. Training step of that size, tables'
// indexing in torch / these kernels: 2894 / 2841 us.
constexpr int64_t kMostBlocks = 0xffffffff / 256;  // blocks of 256 threads: a launch has under 2^32 threads along x
constexpr int kEmbedLds = 64 << 10;
constexpr int64_t kEmbedVocab = 1024;
constexpr int kEmbedBatch = 64;  // rows whose loads go out together, a token per lane

template <typename T, int C>
__global__ __launch_bounds__(64) void embed_bwd_tok_kernel(const int64_t* __restrict__ tokens, const T* __restrict__ dh,
                                                           float* __restrict__ part, int rows, int dim, int vocab,
                                                           int slice, int64_t slab) {
  extern __shared__ float table[];
  const int lane = threadIdx.x, col = (int)blockIdx.x * C + lane, from = min(col, dim - 1);
  const bool on = lane < C && col < dim;
  for (int i = lane; i < vocab * C; i += 64) table[i] = 0.f;
  __syncthreads();
  const int end = min(rows, ((int)blockIdx.y + 1) * slice);
  for (int r = (int)blockIdx.y * slice; r < end; r += kEmbedBatch) {
    T v[kEmbedBatch];
#pragma unroll
    for (int u = 0; u < kEmbedBatch; ++u) v[u] = dh[(int64_t)min(r + u, end - 1) * dim + from];
    int64_t tok = tokens[min(r + lane, end - 1)];
    tok += tok < 0 ? vocab : 0;
    // The forward has refused what is outside the table.
    const int mine = r + lane < end ? (int)max((int64_t)0, min(tok, (int64_t)vocab - 1)) : -1;
#pragma unroll
    for (int u = 0; u < kEmbedBatch; u += 2) {  // two rows to a read of the table where their tokens differ
      // Read with every lane active: the lanes past C hold tokens too.
      const int t0 = __builtin_amdgcn_readlane(mine, u), t1 = __builtin_amdgcn_readlane(mine, u + 1);
      if (!on || t0 < 0) continue;
      const float v0 = Elem<T>::to_f32(v[u]), v1 = t1 < 0 ? 0.f : Elem<T>::to_f32(v[u + 1]);
      float* const p0 = table + t0 * C + lane;
      if (t1 < 0 || t0 == t1) {
        *p0 = *p0 + v0 + v1;
      } else {
        float* const p1 = table + t1 * C + lane;
        const float a = *p0, b = *p1;
        *p0 = a + v0;
        *p1 = b + v1;
      }
    }
  }
  __syncthreads();
  if (!on) return;
  part += blockIdx.y * slab + col;
  for (int i = 0; i < vocab; ++i) part[(int64_t)i * dim] = table[i * C + lane];
}

// The position table's gradient: row s is the sum of dh over the sequences at position s, zero
// past the sequences' length. Four waves take every fourth sequence of 64 columns.
template <typename T, typename TO>
__global__ __launch_bounds__(256) void embed_bwd_pos_kernel(const T* __restrict__ dh, TO* __restrict__ out, int batch,
                                                            int period, int dim) {
  __shared__ float red[3][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int s = blockIdx.x, col = (int)blockIdx.y * 64 + lane;
  float acc = 0.f;
  if (s < period && col < dim) {
#pragma unroll 8
    for (int b = wave; b < batch; b += 4) acc += Elem<T>::to_f32(dh[((int64_t)b * period + s) * dim + col]);
  }
  if (wave > 0) red[wave - 1][lane] = acc;
  __syncthreads();
  if (wave == 0 && col < dim)
    out[(int64_t)s * dim + col] = Elem<TO>::from_f32(acc + red[0][lane] + red[1][lane] + red[2][lane]);
}

struct EmbedBwd {
  int cols, slices, slice;
  int64_t slab;  // floats from one slice's table to the next
};
bool embed_bwd_plan(int64_t rows, int64_t period, int64_t dim, int64_t vocab, int64_t seq, EmbedBwd& p) {
  if (rows < 1 || rows > 0x3fffffff || period < 1 || rows % period || seq < period || seq > kMostBlocks || dim < 1 ||
      dim > 64 * 65535 || vocab < 1 || vocab > kEmbedVocab)
    return false;
  p.cols = vocab <= 256 ? 64 : vocab <= 512 ? 32 : 16;
  p.slices = (int)std::clamp<int64_t>(std::min(512 / cdiv(dim, (int64_t)p.cols), rows / 64), 1, 64);
  p.slice = (int)cdiv(rows, (int64_t)p.slices);
  p.slab = (vocab * dim + 3) / 4 * 4;
  return true;
}

template <typename T, typename TO>
int embed_bwd_launch(const int64_t* tokens, const T* dh, TO* dtok, TO* dpos, int64_t rows, int64_t period, int64_t dim,
                     int64_t vocab, int64_t seq, const EmbedBwd& p, float* part, hipStream_t st) {
  const dim3 grid((unsigned)cdiv(dim, (int64_t)p.cols), (unsigned)p.slices);
  const size_t lds = (size_t)vocab * p.cols * 4;
  static_assert(256 * 64 * 4 == kEmbedLds && 512 * 32 * 4 == kEmbedLds && kEmbedVocab * 16 * 4 == kEmbedLds);
  auto tok = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(64), lds, st, tokens, dh, part, (int)rows, (int)dim, (int)vocab, p.slice, p.slab);
  };
  if (p.cols == 64)
    tok(embed_bwd_tok_kernel<T, 64>);
  else if (p.cols == 32)
    tok(embed_bwd_tok_kernel<T, 32>);
  else
    tok(embed_bwd_tok_kernel<T, 16>);
  const int64_t mn = vocab * dim;
  hipLaunchKernelGGL((gemm_splitk_reduce_kernel<TO>), dim3((unsigned)cdiv(cdiv(mn, (int64_t)4), (int64_t)256)), dim3(256),
                     0, st, part, dtok, mn, p.slices, (bf16*)nullptr, p.slab);
  hipLaunchKernelGGL((embed_bwd_pos_kernel<T, TO>), dim3((unsigned)seq, (unsigned)cdiv(dim, (int64_t)64)), dim3(256), 0, st,
                     dh, dpos, (int)(rows / period), (int)period, (int)dim);
  return check_launch("ferrite_embed_bwd");
}

}  // namespace
}  // namespace ferrite

extern "C" int ferrite_hip_heads_split(const void* tokens, void* const* heads, int64_t b, int64_t s, int64_t groups,
                                       int64_t h, int64_t d, int dtype, void* stream) {
  return ferrite::heads_dispatch<true>("ferrite_hip_heads_split", const_cast<void*>(tokens), heads, b, s, groups, h,
                                       d, dtype, stream);
}

extern "C" int ferrite_hip_heads_merge(void* const* heads, void* tokens, int64_t b, int64_t s, int64_t groups,
                                       int64_t h, int64_t d, int dtype, void* stream) {
  return ferrite::heads_dispatch<false>("ferrite_hip_heads_merge", tokens, heads, b, s, groups, h, d, dtype, stream);
}

extern "C" int ferrite_internal_embed(const int64_t* tokens, const int32_t* pos, const void* tok_emb,
                                      const void* pos_emb, void* out, int64_t rows, int64_t dim, int64_t vocab,
                                      int64_t seq, int64_t period, int emb_dtype, int out_dtype, void* stream) {
  using namespace ferrite;
  const char* name = "ferrite_internal_embed";
  if (!valid_dtype(emb_dtype) || !valid_dtype(out_dtype))
    return fail(FERRITE_ERR_INVALID_ARGUMENT, std::string(name) + ": dtype must be FERRITE_F32 or FERRITE_BF16");
  if (rows < 0 || rows > kMostBlocks || dim < 1 || vocab < 1 || seq < 1 ||
      (rows > 0 && !pos && (period < 1 || period > seq)))
    return fail(FERRITE_ERR_INVALID_ARGUMENT, std::string(name) + ": sizes out of range");
  if (rows == 0) return FERRITE_OK;
  if (!tokens || !tok_emb || !pos_emb || !out)
    return fail(FERRITE_ERR_INVALID_ARGUMENT, std::string(name) + ": null pointer");
  auto go = [&](auto* te, auto* to) {
    typedef std::remove_const_t<std::remove_pointer_t<decltype(te)>> TE;
    typedef std::remove_pointer_t<decltype(to)> TO;
    auto launch = [&](auto kernel, int64_t v) {
      const int64_t threads = std::min<int64_t>(256, cdiv(cdiv(dim, v), (int64_t)64) * 64);
      hipLaunchKernelGGL(kernel, dim3((unsigned)rows), dim3((unsigned)threads), 0, static_cast<hipStream_t>(stream), tokens,
                         pos, te, static_cast<const TE*>(pos_emb), to, dim, vocab, seq, (int)period);
    };
    if (dim % 4 == 0 && al16(tok_emb) && al16(pos_emb) && al16(out))
      launch(embed_kernel<TE, TO, 4>, 4);
    else
      launch(embed_kernel<TE, TO, 1>, 1);
  };
  auto to = [&](auto* te) {
    if (out_dtype == FERRITE_BF16)
      go(te, static_cast<bf16*>(out));
    else
      go(te, static_cast<float*>(out));
  };
  if (emb_dtype == FERRITE_BF16)
    to(static_cast<const bf16*>(tok_emb));
  else
    to(static_cast<const float*>(tok_emb));
  return check_launch(name);
}

extern "C" int64_t ferrite_internal_embed_bwd_workspace(int64_t rows, int64_t period, int64_t dim, int64_t vocab,
                                                        int64_t seq) {
  ferrite::EmbedBwd p;
  return ferrite::embed_bwd_plan(rows, period, dim, vocab, seq, p) ? p.slices * p.slab * 4 : -1;
}

extern "C" int ferrite_internal_embed_bwd(const int64_t* tokens, const void* dh, void* dtok, void* dpos, int64_t rows,
                                          int64_t period, int64_t dim, int64_t vocab, int64_t seq, int dh_dtype,
                                          int emb_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace ferrite;
  const char* name = "ferrite_internal_embed_bwd";
  EmbedBwd p;
  if (!valid_dtype(emb_dtype) || !valid_dtype(dh_dtype))
    return fail(FERRITE_ERR_INVALID_ARGUMENT, std::string(name) + ": dtype must be FERRITE_F32 or FERRITE_BF16");
  if (!embed_bwd_plan(rows, period, dim, vocab, seq, p))
    return fail(FERRITE_ERR_INVALID_ARGUMENT, std::string(name) + ": sizes out of range");
  if (!tokens || !dh || !dtok || !dpos || !workspace || !al16(workspace) || !al16(dtok) ||
      workspace_bytes < p.slices * p.slab * 4)
    return fail(FERRITE_ERR_INVALID_ARGUMENT, std::string(name) + ": null or unaligned pointer, or small workspace");
  auto go = [&](auto* g, auto* d) {
    return embed_bwd_launch(tokens, g, d, static_cast<decltype(d)>(dpos), rows, period, dim, vocab, seq, p,
                            static_cast<float*>(workspace), static_cast<hipStream_t>(stream));
  };
  auto to = [&](auto* g) {
    return emb_dtype == FERRITE_BF16 ? go(g, static_cast<bf16*>(dtok)) : go(g, static_cast<float*>(dtok));
  };
  return dh_dtype == FERRITE_BF16 ? to(static_cast<const bf16*>(dh)) : to(static_cast<const float*>(dh));
}
