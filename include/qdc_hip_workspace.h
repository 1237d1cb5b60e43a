/* qdc_hip_workspace.h -- entry points of libqdc_hip.so that work through a
 * caller's scratch buffer or replace several entry points of qdc_hip.h by one
 * pass.  Types, status codes, dtype codes and stream rules are those of
 * qdc_hip.h: nothing is allocated or kept, everything is enqueued on `stream`,
 * and a negative status is returned before anything is enqueued.
 */
#ifndef QDC_HIP_WORKSPACE_H
#define QDC_HIP_WORKSPACE_H

#include "qdc_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Bytes of 16-byte aligned device scratch that qdc_delta_scan_ws needs for these
 * sizes, or 0 when it has no form for them (call qdc_delta_scan then): key_dim
 * 32, 64 or 128 and value_dim a multiple of 16. */
int64_t qdc_delta_scan_workspace(int64_t batch, int64_t seq, int64_t heads, int64_t key_dim,
                                 int64_t value_dim);

/* The recurrence of qdc_delta_scan, the same arguments and results, as two
 * launches: what does not involve the state is computed for all chunks of 16
 * tokens at once into `workspace` (workspace_bytes >= qdc_delta_scan_workspace),
 * then the state runs over the chunks.  q, k and v must be 16-byte aligned with
 * ld_qk and ld_v multiples of 4 below 2^25 (QDC_ERR_SHAPE otherwise); the workspace may not
 * overlap any other argument. */
int32_t qdc_delta_scan_ws(void *out, int32_t out_dtype, const float *q, const float *k,
                          const float *v, const float *beta, const float *decay, int64_t batch,
                          int64_t seq, int64_t heads, int64_t key_heads, int64_t key_dim,
                          int64_t value_dim, int64_t ld_qk, int64_t ld_v, void *workspace,
                          int64_t workspace_bytes, hipStream_t stream);

/* Causal attention of prepared (normalised, rotated) heads with its output gate:
 *     out[t, h*head_dim + r] = sigmoid(gate[t, h, r]) *
 *         sum_j softmax_j(scale * q[t, h] . k[j, g]) v[j, g, r],  g = h / (heads/kv_heads)
 * over the keys j of the same sequence with j <= t whose mask[b, j] != 0 (mask
 * null: all); a query that sees no key weighs every key of its sequence alike.
 * What qdc_attention_softmax and qdc_attention_gate give around two batched
 * products, with no score matrix.  `dtype` is the type of q, k, v and gate, which
 * are views of rows of head_dim contiguous elements with their strides between
 * tokens and heads in elements; out_dtype may also be QDC_BF16X2.  head_dim 64,
 * 128 or 256; all strides multiples of 16 bytes and all pointers 16-byte aligned
 * (QDC_ERR_SHAPE otherwise).  scale is positive, and scale * log2(e) finite
 * (QDC_ERR_RANGE otherwise; qdc_attention_softmax takes any scale).  out may not
 * overlap any input. */
int32_t qdc_attention_fused(void *out, int32_t out_dtype, const void *q, const void *k,
                            const void *v, const void *gate, const int32_t *mask, int64_t batch,
                            int64_t seq, int64_t heads, int64_t kv_heads, int64_t head_dim,
                            int64_t q_tok, int64_t q_head, int64_t k_tok, int64_t k_head,
                            int64_t v_tok, int64_t v_head, int64_t gate_tok, int64_t gate_head,
                            int64_t out_tok, float scale, int32_t dtype, hipStream_t stream);

/* fp32 sums of out = a w^T for an output of few tiles: the inner dimension is cut
 * into `parts`, and out is [parts][rows][cols], one partial product after the other.
 * `a` is [rows, inner] bf16, or with a_dtype QDC_BF16X2 in the split form (2 inner
 * values a row); `w` is [cols, inner] bf16.  ld_a and ld_w in bf16 values.  inner a
 * multiple of 64 (32 for a split a), cols of 128, strides of 8, parts at most the
 * steps of 64 values of a, pointers 16-byte aligned (QDC_ERR_SHAPE otherwise). */
int32_t qdc_linear_parts(float *out, const void *a, const void *w, int64_t rows, int64_t inner,
                         int64_t cols, int64_t ld_a, int64_t ld_w, int64_t parts, int32_t a_dtype,
                         hipStream_t stream);

/* residual = x + the sum of `parts` [rows, width] tensors and normed = rms(residual) *
 * (1 + norm) * mask (mask null: 1): qdc_residual_rmsnorm(_masked) reading the sums of
 * qdc_linear_parts.  norm is fp32 for out_dtype QDC_F32, else bf16; out_dtype may be
 * QDC_BF16X2; width 256, 512, 1024 or 2048.  residual may be x; otherwise outputs
 * overlap neither each other nor an input. */
int32_t qdc_residual_rms_parts(float *residual, void *normed, const float *x, const float *sums,
                               int64_t parts, const void *norm, const int32_t *mask, int64_t rows,
                               int64_t width, float eps, int32_t out_dtype, hipStream_t stream);

/* An fp32 projection of few rows with the row work around it: out = in w, or with
 * swiglu != 0 and w = [gate | up] of 2 cols columns out = silu(in gate) * (in up), where
 *   input 0: in = a;
 *   input 1: residual = a + b, in = rms(residual) * (1 + norm) * mask (mask null: 1), as
 *            qdc_residual_rmsnorm(_masked); residual is [rows, inner];
 *   input 2: in = the gated norm of every head of head_dim values of a with z = b, as
 *            qdc_gated_rmsnorm; swiglu must be 0.
 * inner 128, 256 or 512, cols a multiple of 64, head_dim of 64 that divides inner; rows
 * ld_a, ld_b, ld_w (of w: [inner, columns]) and ld_out elements apart, multiples of 4;
 * pointers 16-byte aligned (QDC_ERR_SHAPE otherwise; an input outside 0..2
 * QDC_ERR_RANGE).  Pointers an input does not use are ignored.  Outputs overlap
 * neither each other nor an input. */
int32_t qdc_linear_f32(float *out, float *residual, const float *a, const float *b,
                       const float *norm, const int32_t *mask, const float *w, int64_t rows,
                       int64_t inner, int64_t cols, int64_t head_dim, int64_t ld_a, int64_t ld_b,
                       int64_t ld_w, int64_t ld_out, float eps, int32_t input, int32_t swiglu,
                       hipStream_t stream);

#ifdef __cplusplus
}
#endif
#endif
