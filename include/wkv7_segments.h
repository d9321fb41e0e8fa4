/*
 * wkv7_segments.h -- the WKV7 forward and backward (wkv7.h) with a caller's
 * workspace, for calls with few (batch, head) pairs. Operand names, layouts,
 * checks, errors and threading rules are wkv7.h's.
 */
#ifndef RWKV_RS_AMD_WKV7_SEGMENTS_H
#define RWKV_RS_AMD_WKV7_SEGMENTS_H

#include "wkv7.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Calls with few (batch, head) pairs. One workgroup walks a whole sequence of
 * one pair, so such a call leaves most of the GPU idle. Given a workspace,
 * wkv7_forward_ws / wkv7_backward_ws cut each sequence into segments that run
 * side by side: the state is an affine function of an earlier state, so a
 * first pass forms every segment's transition, a second one the states at
 * the segments' boundaries, and the third runs each segment from its own.
 * The arithmetic is the chunked kernels' (above); a boundary state goes
 * through a transition matrix instead of through the steps one by one. No
 * counterpart in the reference.
 *
 * The workspace is device memory of at least wkv7_*_workspace_bytes bytes for
 * the same arguments (0 where the call is not cut: the shape fills the GPU, is
 * too short, or runs on kernels that are not cut; -1 for invalid arguments),
 * 16-byte aligned, overlapping no operand; its contents need no
 * initialisation and mean nothing afterwards, and calls that may overlap in
 * time need one each. With workspace NULL, or fewer bytes than that, the call
 * runs in one piece, as wkv7_forward_ex / wkv7_backward_ex do.
 */
int64_t wkv7_forward_workspace_bytes(int64_t batch_size, int64_t context_len,
                                     int64_t num_heads, int64_t head_size,
                                     int64_t chunk_len, int dtype,
                                     const wkv7_options *options);
int64_t wkv7_backward_workspace_bytes(int64_t batch_size, int64_t context_len,
                                      int64_t num_heads, int64_t head_size,
                                      int64_t chunk_len, int dtype,
                                      const wkv7_options *options);

int wkv7_forward_ws(const void *weight_decay, const void *receptance,
                    const void *key, const void *value, const void *removal,
                    const void *replacement, const float *initial_state,
                    int64_t batch_size, int64_t context_len, int64_t num_heads,
                    int64_t head_size, int64_t chunk_len, int dtype,
                    int use_initial_state, int return_final_state, float *state,
                    float *removal_state, void *output, float *final_state,
                    const wkv7_options *options, void *workspace,
                    int64_t workspace_bytes, void *stream);

int wkv7_backward_ws(const void *weight_decay, const void *receptance,
                     const void *key, const void *value, const void *removal,
                     const void *replacement, const float *state,
                     const float *removal_state, const void *output_grad,
                     const float *final_state_grad, int64_t batch_size,
                     int64_t context_len, int64_t num_heads, int64_t head_size,
                     int64_t chunk_len, int dtype, int use_final_state_grad,
                     int write_initial_state_grad, void *weight_decay_grad,
                     void *receptance_grad, void *key_grad, void *value_grad,
                     void *removal_grad, void *replacement_grad,
                     float *initial_state_grad, const wkv7_options *options,
                     void *workspace, int64_t workspace_bytes, void *stream);

#ifdef __cplusplus
}
#endif

#endif /* RWKV_RS_AMD_WKV7_SEGMENTS_H */
