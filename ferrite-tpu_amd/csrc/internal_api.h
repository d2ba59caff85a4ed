// Entry points of libferrite_hip.so for the Python package of the same tree alone. They keep the
// conventions of ferrite_hip.h (device pointers, sizes, a stream; 0 or a FERRITE_ERR_* code;
// nothing allocated, nothing synchronised), but are no part of its C ABI and change with the
// package.
#pragma once

#include <stdint.h>

extern "C" {

/*
 * The bf16 product for operands the matrix kernel cannot read in place: any M, N, K and
 * any 2-byte aligned pointers, either operand given transposed (as ferrite_hip_matmul_ex).
 * Operands whose rows do not start at 16-byte boundaries are first copied into the
 * workspace with their rows padded to a multiple of 8 elements; the workspace also holds
 * the K split's partials. It has ferrite_internal_matmul_ragged_workspace(...) bytes (0: none
 * needed; -1: sizes out of range, an operand of 2^33 elements or more among them), which
 * depends on the sizes and on the operands' alignment, and is 16-byte aligned; a smaller
 * one fails with FERRITE_ERR_INVALID_ARGUMENT. Its content need not survive the call.
 */
int64_t ferrite_internal_matmul_ragged_workspace(const void* x, const void* y, int64_t m, int64_t n, int64_t k,
                                                 int x_t, int y_t);
/*
 * 1 where that is the faster one, 0 where ferrite_hip_matmul_ex's own choice on untransposed operands is
 * (transposed ones copied first).
 */
int ferrite_internal_matmul_ragged_better(const void* x, const void* y, int64_t m, int64_t n, int64_t k, int x_t,
                                          int y_t);
int ferrite_internal_matmul_ragged(const void* x, const void* y, void* out, int64_t m, int64_t n, int64_t k, int x_t,
                                   int y_t, int out_dtype, void* workspace, int64_t workspace_bytes, void* stream);

/*
 * out[M,N] = x[M,K] . bf16(w[K,N]) (w_t: w holds [N,K]) for a bf16 x and a float w whose
 * elements are rounded to bf16 as they are read (model/gpt.py:95-104, :143: the casts of the
 * linear layers' weights and of the tied head's), with M <= 64 rows and a bf16 or float out.
 * With aux (bf16 out, w not transposed), the GELU epilogue: aux <- bf16(x . w), out <- bf16(gelu(aux)).
 * A workspace of ferrite_internal_linear_f32w_workspace(...) bytes (-1: sizes out of range),
 * 16-byte aligned, lets a deep K split; with less it does not.
 */
int64_t ferrite_internal_linear_f32w_workspace(const void* x, const float* w, int64_t m, int64_t n, int64_t k, int w_t);
int ferrite_internal_linear_f32w(const void* x, const float* w, void* out, void* aux, int64_t m, int64_t n, int64_t k,
                                 int w_t, int out_dtype, void* workspace, int64_t workspace_bytes, void* stream);

/*
 * ferrite_hip_decode_attention with q, k_new and v_new [B, H, D] given with one stride of
 * new_stride >= H * D elements (a multiple of 8) from a sequence to the next, as they lie in a
 * fused projection; the heads of a sequence are dense.
 */
int ferrite_internal_decode_attention(const void* q, const void* k_new, const void* v_new, void* k_cache, void* v_cache,
                                      const int32_t* pos, void* out, int64_t b, int64_t h, int64_t max_len, int64_t d,
                                      int64_t new_stride, int dtype, float scale, void* workspace,
                                      int64_t workspace_bytes, void* stream);

/*
 * out[r] = tok_emb[tokens[r]] + pos_emb[pos[r]] for one token per row (model/gpt.py:124-127 at the
 * positions of a decode step; without pos, row r is at position r % period, period <= seq),
 * summed and rounded in emb_dtype, then converted to out_dtype.
 * tok_emb [vocab, dim], pos_emb [seq, dim]. A negative index counts from the table's end; one
 * outside the table traps, as the gather of a tensor library does.
 */
int ferrite_internal_embed(const int64_t* tokens, const int32_t* pos, const void* tok_emb, const void* pos_emb, void* out,
                           int64_t rows, int64_t dim, int64_t vocab, int64_t seq, int64_t period, int emb_dtype,
                           int out_dtype, void* stream);

/*
 * Its gradients without pos, summed in f32 in a fixed order: dtok[vocab, dim], the rows of
 * dh[rows, dim] summed by token, and dpos[seq, dim], by position (zero from period on). Up to 1024
 * tokens in the vocabulary and whole sequences. The workspace, 16-byte aligned as dtok is, has
 * ferrite_internal_embed_bwd_workspace(...) bytes (-1: sizes out of range).
 */
int64_t ferrite_internal_embed_bwd_workspace(int64_t rows, int64_t period, int64_t dim, int64_t vocab, int64_t seq);
int ferrite_internal_embed_bwd(const int64_t* tokens, const void* dh, void* dtok, void* dpos, int64_t rows,
                               int64_t period, int64_t dim, int64_t vocab, int64_t seq, int dh_dtype, int emb_dtype,
                               void* workspace, int64_t workspace_bytes, void* stream);

}  // extern "C"
