// Entry points of the package's own model layers (asrback_amd/*.py): the
// element-wise work around the attention calls of asrattn.h.  Not part of
// the C ABI that replaces the reference's attention ops; the same
// conventions hold (device pointers, element strides, a stream, no
// allocation, no synchronization, asrattn_last_error for messages).
#pragma once

#include <stdint.h>

#include "asrattn.h"

extern "C" {

// The rows a prompt pass prepares for its attention: per-head RMSNorm and
// rotary embedding of the queries and keys, the values' RMSNorm without
// weights (v_norm), and the writes of keys and values to the cache.
//
//   q' = rot(norm(q, q_norm), cos, sin)     -> q_out
//   k' = rot(norm(k, k_norm), cos, sin)     -> k_out and the cache
//   v' = norm(v, 1) (v_norm != 0; else v)   -> v_out (if given) and the cache
//
// with asrattn_decode_append's norm and rot, rounded in the element type as
// the reference's ops round.  Token t of sequence b (batch x tokens of them)
// is row b * tokens + t of the outputs, which are contiguous.  Its cache slot
// is (rows[b * tokens + t], positions[b * tokens + t]), or (rows[b], t) with
// positions NULL; negative indices count from the end, and slots outside the
// cache are not written.  With a block table (int32, bt_stride entries per
// cache row) the slot lies in page block_table[row][position / page_size]
// of the pool, or in the sink page num_pages where that is outside [0,
// num_pages).  k NULL: queries only.
typedef struct asrlayer_prompt_params {
  const void *q, *k, *v;
  void *q_out, *k_out, *v_out;
  void *k_cache, *v_cache;
  int64_t q_batch_stride, q_token_stride, q_head_stride;
  int64_t k_batch_stride, k_token_stride, k_head_stride;
  int64_t v_batch_stride, v_token_stride, v_head_stride;
  // Cache: row (paged: page), position and head strides, and its extent.
  int64_t kc_row_stride, kc_pos_stride, kc_head_stride;
  int64_t vc_row_stride, vc_pos_stride, vc_head_stride;
  int64_t cache_rows, cache_length;
  const int64_t *rows, *positions;
  const int32_t* block_table;
  int64_t bt_stride;
  int32_t page_size, num_pages;
  const void *q_norm, *k_norm;  // (head_dim,)
  const void *cos, *sin;        // (batch, tokens, head_dim) by the strides below
  int64_t rope_batch_stride, rope_token_stride;
  float q_eps, k_eps, v_eps;
  int32_t v_norm;
  int32_t batch, tokens, heads_q, heads_kv, head_dim, dtype;
} asrlayer_prompt_params;

int asrlayer_prompt_rows(const asrlayer_prompt_params* params, void* stream);

// Linear layers over the few rows of a decoder step:
//
//   out[i] = act(norm(x) w[i]^T + b[i])             (i < 3, n[i] > 0)
//   out[i] = residual + (norm(x) w[i]^T + b[i])     (residual given)
//
// with norm the layer norm over the k inputs (ln_weight NULL: none), sums in
// float32 and each result rounded in the element type where the separate
// torch ops round: after the norm, after the product and bias, after the
// activation, after the residual sum.  x: (rows, k), rows x_row_stride
// apart; w[i]: (n[i], k), contiguous; b[i]: (n[i]) or NULL; out[i]: (rows,
// n[i]), contiguous; residual: (rows, n[0]), with one matrix.  act 0: none,
// 1: gelu (exact).  rows 1 .. 16; k a multiple of 16 bytes and at most 1024
// times that.
typedef struct asrlayer_linear_params {
  const void* x;
  int64_t x_row_stride;
  const void *ln_weight, *ln_bias;
  const void* w[3];
  const void* b[3];
  void* out[3];
  const void* residual;
  int64_t r_row_stride;
  float ln_eps;
  int32_t n[3];
  int32_t rows, k, act, dtype;
} asrlayer_linear_params;

int asrlayer_rows_linear(const asrlayer_linear_params* params, void* stream);

// A decoder step's input: out[r] = token_weight[tokens[r * token_stride]] +
// position_weight[positions[r]], tables (vocab, width) and (length, width), all
// contiguous; rows whose token or position lies outside are NaN.  width a
// multiple of 16 bytes.
typedef struct asrlayer_embed_params {
  const void *token_weight, *position_weight;
  const int64_t *tokens, *positions;
  void* out;
  int64_t token_stride, vocab, length;
  int32_t rows, width, dtype;
} asrlayer_embed_params;

int asrlayer_embed_rows(const asrlayer_embed_params* params, void* stream);

// A linear layer over bf16 rows (batch x rows of k inputs, n outputs each):
//
//   out[b, t, :] = x[b, t, :] w^T + bias        (accumulate 0; bias or NULL)
//   out[b, t, :] = out[b, t, :] + x[b, t, :] w^T    (accumulate 1, no bias)
//
// with float32 sums, rounded once.  w (n, k) contiguous; rows x_row_stride
// and out_row_stride apart.  used (int32[batch], device, or NULL): rows t >=
// used[b] are neither read nor written.  k a multiple of 64, n of 8.
typedef struct asrlayer_gemm_params {
  const void *x, *w, *bias;
  void* out;
  const int32_t* used;
  int64_t x_batch_stride, x_row_stride, out_batch_stride, out_row_stride;
  int32_t batch, rows, n, k, accumulate;
} asrlayer_gemm_params;

int asrlayer_gemm(const asrlayer_gemm_params* params, void* stream);

}  // extern "C"
