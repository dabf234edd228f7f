/*
 * e2h_seq.h -- C ABI of libe2h_seq.so: the kernels of decoder layers that carry per-sequence state beside a KV cache
 * (windowed attention with kept first tokens, rotation and sinks, HGRN2, gated delta rule, causal convolutions over time) and
 * of mixtures of experts, for AMD MI355X (gfx950).
 *
 * Conventions
 *   - every pointer is a DEVICE pointer into memory the caller owns; nothing here allocates, frees or synchronises.
 *     Kernels are enqueued on `stream` (a hipStream_t passed as void*) and may be recorded into a HIP graph.
 *   - activations are bfloat16 or float32 (`dtype`: E2H_SEQ_BF16 / E2H_SEQ_F32); norms, biases, gates, convolution
 *     weights of the norm kernels, the residual stream and recurrent state are float32 in both cases.
 *   - a call covers `seqlen` consecutive tokens of each of `batch` sequences; row b * seqlen + t is token t of sequence b.
 *     `input_pos` points at the position of token 0 (int64, device memory: graph replays move it), `first` (NULL = all
 *     zero) at one int64 per sequence: positions before it are padding and do not exist for the sequence.
 *   - state is continued from the previous call when the position is not 0 and taken as empty when it is.
 *   - the convolutions keep their last inputs in a ring of `taps` slots, slot = position mod taps.  With seqlen == 1 the
 *     kernel puts the new input into tail_out, which may be tail_in itself; with seqlen > 1 tail_out must be different
 *     memory, receives the last taps - 1 inputs, and the caller copies it over tail_in afterwards.
 *   - every entry point returns E2H_OK or a negative E2H_ERR_* code of e2h_quant.h; sizes that a kernel does not take give
 *     E2H_ERR_BAD_SHAPE.
 */
#ifndef E2H_SEQ_H
#define E2H_SEQ_H

#include <stdint.h>

#include "e2h_quant.h"

#ifdef __cplusplus
extern "C" {
#endif

#define E2H_SEQ_ABI_VERSION 2
#define E2H_SEQ_BF16 0
#define E2H_SEQ_F32 1

int e2h_seq_abi_version(void);
/* Experiment switches (0 = built-in choice): "recurrence_form" 1 = token by token, 2 = chunked; "recurrence_chunk" = tokens a
 * workgroup of the chunked HGRN2 form covers; "norm_run" = tokens a workgroup of the norm kernel covers where it convolves;
 * "attention_decode_waves" = 4 or 8; "attention_prompt_queries" = 64 or 128 a workgroup of the prompt kernels takes; "expert_form" 1 = the plain kernel for all sizes, 2 = expert lists made inside the matmul
 * (few rows), 3 = sorted rows in large tiles. */
int e2h_seq_set_option(const char *name, int value);

/* x_out = x + norm(d); h = norm(x_out); out = h + conv(h), each step optional:
 *   d = delta + sum_k term_weights[row, k] * terms[row * n_terms + k]   (either part may be absent)
 *   RMS norm:   norm(z) = z / sqrt(mean(z^2) + eps) * (offset + weight)
 *   layer norm: norm(z) = (z - mean(z)) / sqrt(mean((z - mean(z))^2) + eps) * (offset + weight) + bias
 *   conv(h)[t] = sum_j w[j, :] h[t - taps + 1 + j], zero before the sequence starts.
 * delta and terms NULL: x_out = x, not stored.  norm_weight NULL: h = x_out.  conv NULL: out = h.  One of x_out and out may be
 * NULL.  Layer norms and terms come without conv. */
#define E2H_SEQ_RMS_NORM 0
#define E2H_SEQ_LAYER_NORM 1
typedef struct {
  int32_t dtype; /* of delta and out */
  int32_t taps;
  int64_t batch, seqlen, width;
  float eps, delta_offset, norm_offset;
  int32_t norm_kind;         /* of both norms */
  const float *x;            /* [rows, width] */
  const void *delta;         /* [rows, width] or NULL */
  const float *delta_weight; /* [width] */
  float *x_out;              /* [rows, width], different memory from x when seqlen > 1 */
  const float *norm_weight;  /* [width] or NULL */
  const float *conv;         /* [taps, width] or NULL; the last row is the current token's */
  const float *tail_in;      /* [batch, taps, width] */
  float *tail_out;
  void *out;                 /* [rows, width] */
  const int64_t *input_pos;
  const int64_t *first;
  const float *delta_bias, *norm_bias; /* [width] or NULL, layer norm only */
  const void *terms;                   /* [rows * n_terms, width] or NULL */
  const float *term_weights;           /* [rows, n_terms] */
  int64_t n_terms;
} e2h_norm_conv_args;
int e2h_seq_norm_conv(const e2h_norm_conv_args *a, void *stream);
/* The same for one token per sequence, RMS norms and no terms, with delta (NULL in a) the sum in order of `slices` (1 to 4) float32 parts [slices, rows, width], rounded to dtype. */
int e2h_seq_norm_conv_sums(const e2h_norm_conv_args *a, const float *sums, int slices, void *stream);

/* y = act(x w^T) for the few rows of a decode step: x [rows, k], w [n, k] (nn.Linear.weight), y [rows, n], all bfloat16 and contiguous,
 * x and w 16-byte aligned; 1 <= rows <= 64, k a multiple of 8.  Sums are float32; the sum is rounded to bfloat16 before the activation
 * and after it.  act: E2H_SEQ_ACT_NONE, E2H_SEQ_ACT_SQUARE_RELU, or E2H_SEQ_ACT_SOFTCAP with cap > 0.  Some shapes need scratch memory of
 * e2h_seq_linear_scratch_bytes (4-byte aligned; 0: none, negative: the shape is refused). */
#define E2H_SEQ_ACT_NONE 0
#define E2H_SEQ_ACT_SQUARE_RELU 1
#define E2H_SEQ_ACT_SOFTCAP 2
int64_t e2h_seq_linear_scratch_bytes(int64_t rows, int64_t n, int64_t k);
int e2h_seq_linear(const void *x, const void *w, void *y, int64_t rows, int64_t n, int64_t k, int act, float cap, void *scratch,
                   int64_t scratch_bytes, void *stream);

/* The float32 sums of e2h_seq_linear's four slices of K, sums [4, rows, n], for e2h_seq_norm_conv_sums to add; E2H_ERR_BAD_SHAPE where e2h_seq_linear_scratch_bytes is 0. */
int e2h_seq_linear_sums(const void *x, const void *w, float *sums, int64_t rows, int64_t n, int64_t k, void *stream);

/* e2h_seq_linear and e2h_seq_gelu_gate_rows (below) on its result in one launch, bit for bit; E2H_ERR_BAD_SHAPE where e2h_seq_linear_scratch_bytes is not 0. */
int e2h_seq_linear_gelu_gate(const void *x, const void *w, const void *table, const int64_t *tokens, void *y, int64_t rows, int64_t n, int64_t k, int64_t ld, int64_t column,
                             int64_t table_rows, void *stream);

/* The same over many rows (a soft cap between 2^-6 and 2^10): n a multiple of 8, k of 64 and at least 192, x, w and 256 rows of y below 4 GB, all three 16-byte
 * aligned; no scratch.  e2h_seq_linear_rows_pays: 1 where that is expected to take less time than a library product followed by e2h_seq_square_relu or e2h_seq_softcap, else 0. */
int e2h_seq_linear_rows_pays(int64_t rows, int64_t n, int64_t k, int act, float cap);
int e2h_seq_linear_rows(const void *x, const void *w, void *y, int64_t rows, int64_t n, int64_t k, int act, float cap, void *stream);

/* Elementwise steps.  square_relu: y = max(x, 0)^2.  softcap: y = cap tanh(x / cap).  x and y may be the same memory.
 * gelu_gate_rows: y[r, i] = gelu_tanh(gate[r, i]) * table[tokens[r], column + i], i < dim; table rows are ld values long. */
int e2h_seq_square_relu(int dtype, const void *x, void *y, int64_t n, void *stream);
int e2h_seq_softcap(int dtype, const void *x, void *y, int64_t n, float cap, void *stream);
int e2h_seq_gelu_gate_rows(int dtype, const void *gate, const void *table, const int64_t *tokens, void *y, int64_t rows, int64_t dim,
                           int64_t ld, int64_t column, int64_t table_rows, void *stream);
/* embed_rows: x[r, i] = table[tokens[r], i] as float32 and, unless h is NULL, h[r, i] as it is; bfloat16 table [table_rows, width], width % 8 == 0, everything but tokens 16-byte
 * aligned.  Rows of tokens outside the table are no numbers. */
int e2h_seq_embed_rows(const void *table, const int64_t *tokens, float *x, void *h, int64_t rows, int64_t width, int64_t table_rows, void *stream);

/* table[row, i] = (cos, sin) of the turn fraction of position * turns[i], i < pairs: turns[i] is the rotation per position in whole
 * turns (angle / 2 pi), positions count from the sequence's first one.  table is float32 [batch * seqlen, pairs, 2]. */
int e2h_seq_rotary_table(const double *turns, const int64_t *input_pos, const int64_t *first, float *table, int64_t batch, int64_t seqlen,
                         int64_t pairs, void *stream);

/* Softmax attention of each sequence's new tokens over its cache: position i sees j <= i with i - j < window (window 0: no
 * limit) or j < keep_first, counted from the sequence's first position.  The new tokens' keys and values are appended to
 * the caches first.  Query head h reads key/value head h / (heads / kv_heads).  Biases (NULL = none) are added to the projections;
 * the result is out_scale * attention * sigmoid(gate) (no gate when g_off < 0), written at out + row * ld_out + out_off.
 * Each of the following is left out when its pointer is NULL: q_norm, k_norm = RMS norm of every query / key head; rotary = after
 * the norms, the pairs (2 i, 2 i + 1) of queries and keys, i < rot_pairs, are turned by the row's (cos, sin) of e2h_seq_rotary_table; sink
 * = exp(sink[h]) joins the softmax sum of head h, without a value.
 * k_off and v_off both < 0: the layer has no keys of its own and reads the caches as they are. */
typedef struct {
  int32_t dtype;
  int32_t pad_;
  int64_t batch, seqlen, heads, kv_heads, dim, vdim, cache_len;
  const void *proj; /* [rows, ld]: q, k, v, gate at columns q_off, k_off, v_off, g_off */
  int64_t ld, q_off, k_off, v_off, g_off;
  const float *q_bias, *k_bias, *v_bias;
  void *k_cache, *v_cache; /* [batch, kv_heads, cache_len, dim | vdim] */
  const int64_t *input_pos;
  const int64_t *first;
  int64_t window, keep_first;
  float scale, out_scale;
  void *out;
  int64_t ld_out, out_off;
  const float *q_norm, *k_norm; /* [dim] */
  const float *rotary;          /* [batch * seqlen, rot_pairs, 2] */
  int64_t rot_pairs;
  const float *sink; /* [heads] */
  float norm_eps;
  int32_t pad2_;
} e2h_window_attention_args;
int e2h_seq_window_attention(const e2h_window_attention_args *a, void *stream);

/* The same for callers with scratch memory: one-token calls of few sequences share their keys among several workgroups, whose sums meet in
 * scratch_bytes of it (4-byte aligned; e2h_seq_window_attention_scratch_bytes says how many are used, 0: none, negative: the call is
 * refused).  With less, or NULL, they run as above. */
int64_t e2h_seq_window_attention_scratch_bytes(const e2h_window_attention_args *a);
int e2h_seq_window_attention_split(const e2h_window_attention_args *a, void *scratch, int64_t scratch_bytes, void *stream);

/* HGRN2.  Per head: q = silu(q_proj), f = lower + (1 - lower) sigmoid(f_proj + f_bias), S = diag(f) S + (1 - f) v^T,
 * o = S^T q; result out_scale * o / rms(o) * norm_weight at out + row * ld_out + out_off. */
typedef struct {
  int32_t dtype;
  float eps;
  int64_t batch, seqlen, heads, dim, vdim;
  const void *proj;
  int64_t ld, q_off, f_off, v_off;
  const float *f_bias, *lower; /* [heads * dim] */
  const float *norm_weight;    /* [vdim] */
  float *state;                /* [batch, heads, dim, vdim] */
  const int64_t *input_pos;
  const int64_t *first;
  void *scratch;
  int64_t scratch_bytes; /* e2h_seq_hgrn2_scratch_bytes() */
  float out_scale;
  int32_t pad_;
  void *out;
  int64_t ld_out, out_off;
} e2h_hgrn2_args;
int64_t e2h_seq_hgrn2_scratch_bytes(const e2h_hgrn2_args *a);
int e2h_seq_hgrn2(const e2h_hgrn2_args *a, void *stream);

/* Gated delta rule.  q, k (kv_heads x dim) and v (heads x vdim) pass a causal convolution over time and silu; q and k become
 * unit vectors, q is scaled by dim^-1/2; beta = sigmoid(b), g = exp(-exp(A_log) softplus(a + dt_bias)).
 * Per head: S = g S, u = beta (v - S^T k), S = S + k u^T, o = S^T q; result o / rms(o) * norm_weight * silu(gate). */
typedef struct {
  int32_t dtype;
  int32_t taps;
  int64_t batch, seqlen, heads, kv_heads, dim, vdim;
  const void *proj;
  int64_t ld, q_off, k_off, v_off, b_off, a_off, g_off;
  const float *conv; /* [2 kv_heads dim + heads vdim, taps], channels in the order q, k, v */
  const void *tail_in; /* [batch, taps, channels], activations' dtype */
  void *tail_out;
  const float *a_log, *dt_bias, *norm_weight;
  float *state; /* [batch, heads, dim, vdim] */
  const int64_t *input_pos;
  const int64_t *first;
  void *scratch;
  int64_t scratch_bytes; /* e2h_seq_delta_scratch_bytes() */
  float eps, out_scale;
  void *out;
  int64_t ld_out, out_off;
} e2h_delta_args;
/* Prompts of 24 tokens and more hold queries, keys, and a product of either with a chunk's system by whole chunks of 64 tokens and tiles of 16 channels: 474 MB for 8192 tokens of
 * 32 heads (16 key heads) of 128, 3.1 GB for 1024 sequences of 24 such tokens. */
int64_t e2h_seq_delta_scratch_bytes(const e2h_delta_args *a);
int e2h_seq_delta(const e2h_delta_args *a, void *stream);

/* Router of a mixture of experts: logits = router x + bias in float32, the `top` largest of a row are chosen (the lower index
 * of equal ones) in falling order, weights = softmax over the chosen logits.  logits is scratch of rows * experts floats. */
typedef struct {
  int32_t dtype; /* of x and router */
  int32_t pad_;
  int64_t rows, width, experts, top;
  const void *x;      /* [rows, width] */
  const void *router; /* [experts, width] */
  const float *bias;  /* [experts] or NULL */
  float *logits;      /* [rows, experts] */
  int32_t *chosen;    /* [rows, top] */
  float *weights;     /* [rows, top] */
} e2h_route_args;
int e2h_seq_route(const e2h_route_args *a, void *stream);

/* Experts of squared-ReLU feed-forwards: out[row * top + k] = down[e] relu(up[e] x[row])^2 with e = chosen[row, k].  The caller (or
 * e2h_seq_norm_conv's terms) weighs and adds them.  A shared expert (shared_up NULL = none) runs on every row into shared_out.
 * Indices outside 0 .. experts - 1 give rows that are not written. */
typedef struct {
  int32_t dtype;
  int32_t pad_;
  int64_t rows, width, experts, top, ff, shared_ff;
  const void *x;                       /* [rows, width] */
  const int32_t *chosen;               /* [rows, top] */
  const void *up, *down;               /* [experts, ff, width], [experts, width, ff] */
  const void *shared_up, *shared_down; /* [shared_ff, width], [width, shared_ff] */
  void *out;                           /* [rows * top, width] */
  void *shared_out;                    /* [rows, width] */
  void *scratch;
  int64_t scratch_bytes; /* e2h_seq_experts_scratch_bytes() */
} e2h_experts_args;
int64_t e2h_seq_experts_scratch_bytes(const e2h_experts_args *a);
int e2h_seq_experts(const e2h_experts_args *a, void *stream);

#ifdef __cplusplus
}
#endif

#endif
