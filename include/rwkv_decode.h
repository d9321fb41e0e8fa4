/*
 * rwkv_decode.h -- one decode step (context_len 1) of a whole RWKV-7 cell, and
 * of the model's head, for a small batch of sequences. Statuses, dtype codes
 * and threading rules are wkv7.h's.
 *
 * What it computes is the composition of the framework's modules under bf16
 * autocast with fp32 parameters (rwkv-nn cells/causal.rs:166-268, modules/
 * time_mixer/mod.rs:153-217, modules/channel_mixer/mod.rs:83-121): layer norms
 * and the residual stream in fp32; every matrix product from bf16 operands
 * (the weights rounded as they are read) with fp32 sums, its result rounded to
 * bf16; the element-wise ends as in rwkv_neighbors.h, the recurrence as in
 * wkv7.h's wkv7_infer_forward. Intermediate roundings are the modules'; only
 * the order of sums differs.
 */
#ifndef RWKV_RS_AMD_RWKV_DECODE_H
#define RWKV_RS_AMD_RWKV_DECODE_H

#include "wkv7.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Sequences a call may have (four tiles of the 16 rows of a matrix product), and
 * the widest embedding (a norm's 256 threads hold a row, 32 channels each). */
#define RWKV_DECODE_MAX_ROWS 64
#define RWKV_DECODE_MAX_DIM 8192

/* A cell's parameters: fp32, contiguous, 16-byte aligned; C = num_heads * 64.
 * Linear weights are [out, in], LoRA factors [in, out]. LoRA ranks are
 * multiples of 32. The value-residual LoRA is NULL in the first cell. */
typedef struct rwkv_decode_cell_params {
  const float *norm_time_weight, *norm_time_bias;       /* [C] */
  const float *norm_channel_weight, *norm_channel_bias; /* [C] */
  /* token-shift scales [C]: receptance, weight decay, key, value, learning
   * rate, gate */
  const float *mix[6];
  const float *receptance, *key, *value, *output;       /* [C, C] */
  const float *decay_a, *decay_b, *decay_bias;
  const float *rate_a, *rate_b, *rate_bias;
  const float *residual_a, *residual_b, *residual_bias;
  const float *gate_a, *gate_b;
  const float *key_removal, *key_replacement;           /* [C] */
  const float *bonus;                                   /* [num_heads, 64] */
  const float *group_norm_weight, *group_norm_bias;     /* [C] */
  const float *channel_mix;                             /* [C] */
  const float *channel_key;                             /* [4C, C] */
  const float *channel_value;                           /* [C, 4C] */
  int64_t decay_rank, rate_rank, residual_rank, gate_rank;
  float norm_time_eps, norm_channel_eps, group_norm_eps;
} rwkv_decode_cell_params;

/* Device memory a call of `rows` sequences needs, in bytes (16-byte aligned,
 * no initialisation), or -1 for a shape that is not supported. One workspace
 * serves the cells of a step in order: the first cell leaves its value rows
 * in it, which the later cells read. */
int64_t rwkv_decode_workspace_bytes(int64_t rows, int64_t num_heads);

/* One cell. x [rows, C] (fp32, the residual stream) is updated in place. Row b
 * works on slot batch_ids[b] of state ([full_batch, num_heads, 64, 64] in
 * state_dtype, updated in place) and of the token shifts ([full_batch, C]
 * fp32: read from shift_*_in, written whole to shift_*_out, another buffer;
 * other slots are copied). batch_ids must be distinct, so more rows than slots
 * are refused (WKV7_ERR_SHAPE); a row whose id is out of range works on zeros
 * and touches no slot. What a call writes may overlap neither each other nor
 * what it reads (WKV7_ERR_OVERLAP). use_dither and elapsed_t as in
 * wkv7_infer_forward. params->residual_a == NULL marks the first cell. */
int rwkv_decode_cell(const rwkv_decode_cell_params *params, float *x,
                     const int32_t *batch_ids, void *state,
                     const float *shift_time_in, float *shift_time_out,
                     const float *shift_channel_in, float *shift_channel_out,
                     const int32_t *elapsed_t, int64_t rows, int64_t num_heads,
                     int64_t full_batch, int state_dtype, int use_dither,
                     void *workspace, int64_t workspace_bytes, void *stream);

/* The head: logits [rows, vocab] (bf16) = layer norm of x times the
 * unembedding [vocab, C]. */
int rwkv_decode_head(const float *x, const float *norm_weight,
                     const float *norm_bias, float norm_eps,
                     const float *unembed, int64_t rows, int64_t num_heads,
                     int64_t vocab, void *logits, void *workspace,
                     int64_t workspace_bytes, void *stream);

#ifdef __cplusplus
}
#endif

#endif /* RWKV_RS_AMD_RWKV_DECODE_H */
