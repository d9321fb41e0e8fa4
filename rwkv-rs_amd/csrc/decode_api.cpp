// C ABI of the decode step (include/rwkv_decode.h): argument checks, before
// any HIP call, and dispatch.
#include "decode_launch.hpp"

#include <cmath>
#include <initializer_list>

#include "wkv7_launch.hpp"

namespace {

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

bool supported(int64_t rows, int64_t H) {
  return rows >= 0 && rows <= RWKV_DECODE_MAX_ROWS && H > 0 && H * 64 <= RWKV_DECODE_MAX_DIM;
}
// the LoRAs' hidden rows share 4 C of the workspace
bool ranks_fit(const rwkv_decode_cell_params& p, int64_t C) {
  int64_t sum = 0;
  for (int64_t r : {p.decay_rank, p.rate_rank, p.gate_rank, p.residual_a ? p.residual_rank : int64_t(0)}) {
    if (r < 0 || r % 32 != 0 || r > C) return false;
    sum += r;
  }
  return p.decay_rank > 0 && p.rate_rank > 0 && p.gate_rank > 0 && (!p.residual_a || p.residual_rank > 0) &&
         sum <= 4 * C;
}
bool eps_ok(float e) { return e >= 0.f && std::isfinite(e); }

int check_pointers(std::initializer_list<const void*> ps) {
  for (const void* p : ps) {
    if (!p) return WKV7_ERR_NULL_POINTER;
    if (!aligned16(p)) return WKV7_ERR_ALIGNMENT;
  }
  return WKV7_OK;
}

}  // namespace

extern "C" {

int64_t rwkv_decode_workspace_bytes(int64_t rows, int64_t num_heads) {
  return supported(rows, num_heads) ? rwkv_decode::workspace_bytes(rows, num_heads) : -1;
}

int rwkv_decode_cell(const rwkv_decode_cell_params* params, float* x, const int32_t* batch_ids, void* state,
                     const float* shift_time_in, float* shift_time_out, const float* shift_channel_in,
                     float* shift_channel_out, const int32_t* elapsed_t, int64_t rows, int64_t num_heads,
                     int64_t full_batch, int state_dtype, int use_dither, void* workspace,
                     int64_t workspace_bytes, void* stream) {
  if (state_dtype != WKV7_DTYPE_F32 && state_dtype != WKV7_DTYPE_BF16) return WKV7_ERR_DTYPE;
  // distinct ids need as many slots, as in wkv7_infer_forward
  if (!supported(rows, num_heads) || full_batch < rows || full_batch > INT32_MAX - RWKV_DECODE_MAX_ROWS)
    return WKV7_ERR_SHAPE;
  if (use_dither != 0 && use_dither != 1) return WKV7_ERR_FLAGS;
  if (use_dither && state_dtype == WKV7_DTYPE_F32) return WKV7_ERR_FLAGS;
  if (!params) return WKV7_ERR_NULL_POINTER;
  const rwkv_decode_cell_params& p = *params;
  if (!ranks_fit(p, num_heads * 64)) return WKV7_ERR_SHAPE;
  if (!eps_ok(p.norm_time_eps) || !eps_ok(p.norm_channel_eps) || !eps_ok(p.group_norm_eps)) return WKV7_ERR_SHAPE;
  if (int rc = check_pointers({p.norm_time_weight, p.norm_time_bias, p.norm_channel_weight, p.norm_channel_bias,
                               p.mix[0], p.mix[1], p.mix[2], p.mix[3], p.mix[4], p.mix[5], p.receptance, p.key,
                               p.value, p.output, p.decay_a, p.decay_b, p.decay_bias, p.rate_a, p.rate_b,
                               p.rate_bias, p.gate_a, p.gate_b, p.key_removal, p.key_replacement, p.bonus,
                               p.group_norm_weight, p.group_norm_bias, p.channel_mix, p.channel_key,
                               p.channel_value}))
    return rc;
  if (p.residual_a)
    if (int rc = check_pointers({p.residual_a, p.residual_b, p.residual_bias})) return rc;
  if (rows == 0) return WKV7_OK;
  if (int rc = check_pointers({x, state, shift_time_in, shift_time_out, shift_channel_in, shift_channel_out, workspace}))
    return rc;
  if (!batch_ids || (use_dither && !elapsed_t)) return WKV7_ERR_NULL_POINTER;
  if (shift_time_in == shift_time_out || shift_channel_in == shift_channel_out) return WKV7_ERR_OVERLAP;
  if (workspace_bytes < rwkv_decode::workspace_bytes(rows, num_heads)) return WKV7_ERR_SHAPE;
  rwkv_decode::CellCall c{};
  c.p = params;
  c.x = x;
  c.batch_ids = batch_ids;
  c.state = state;
  c.shift_time_in = shift_time_in;
  c.shift_time_out = shift_time_out;
  c.shift_channel_in = shift_channel_in;
  c.shift_channel_out = shift_channel_out;
  c.elapsed_t = elapsed_t;
  c.rows = static_cast<int>(rows);
  c.H = static_cast<int>(num_heads);
  c.full_batch = static_cast<int>(full_batch);
  c.state_bf16 = state_dtype == WKV7_DTYPE_BF16;
  c.use_dither = use_dither;
  c.workspace = workspace;
  return wkv7::hip_status(rwkv_decode::launch_cell(c, static_cast<hipStream_t>(stream)));
}

int rwkv_decode_head(const float* x, const float* norm_weight, const float* norm_bias, float norm_eps,
                     const float* unembed, int64_t rows, int64_t num_heads, int64_t vocab, void* logits,
                     void* workspace, int64_t workspace_bytes, void* stream) {
  if (!supported(rows, num_heads) || vocab <= 0 || vocab > INT32_MAX - 16) return WKV7_ERR_SHAPE;
  if (!eps_ok(norm_eps)) return WKV7_ERR_SHAPE;
  if (int rc = check_pointers({norm_weight, norm_bias, unembed})) return rc;
  if (rows == 0) return WKV7_OK;
  if (int rc = check_pointers({x, logits, workspace})) return rc;
  if (workspace_bytes < rwkv_decode::workspace_bytes(rows, num_heads)) return WKV7_ERR_SHAPE;
  rwkv_decode::HeadCall c{};
  c.x = x;
  c.norm_weight = norm_weight;
  c.norm_bias = norm_bias;
  c.eps = norm_eps;
  c.unembed = unembed;
  c.rows = static_cast<int>(rows);
  c.H = static_cast<int>(num_heads);
  c.vocab = vocab;
  c.logits = static_cast<rwkv_decode::bf16_t*>(logits);
  c.workspace = workspace;
  return wkv7::hip_status(rwkv_decode::launch_head(c, static_cast<hipStream_t>(stream)));
}

}  // extern "C"
