// C ABI of the decode step (include/rwkv_decode.h): argument checks, before
// any HIP call, and dispatch.
#include "decode_launch.hpp"

#include <cmath>
#include <initializer_list>

#include "wkv7_launch.hpp"

namespace {

bool aligned(const void* p, uintptr_t to) { return (reinterpret_cast<uintptr_t>(p) & (to - 1)) == 0; }

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

struct Range {
  const void* p;
  int64_t bytes;
};
typedef std::initializer_list<Range> Ranges;

// each there and 16-byte aligned
int check_pointers(Ranges rs) {
  for (const Range& r : rs) {
    if (!r.p) return WKV7_ERR_NULL_POINTER;
    if (!aligned(r.p, 16)) return WKV7_ERR_ALIGNMENT;
  }
  return WKV7_OK;
}

bool overlaps(const Range& x, const Range& y) {
  if (!x.p || !y.p) return false;
  const auto a = reinterpret_cast<uintptr_t>(x.p), b = reinterpret_cast<uintptr_t>(y.p);
  return a < b + static_cast<uintptr_t>(y.bytes) && b < a + static_cast<uintptr_t>(x.bytes);
}
bool any_overlap(Ranges outs, Ranges ins) {
  for (const Range& o : outs)
    for (const Range& i : ins)
      if (overlaps(o, i)) return true;
  return false;
}
// what a call writes may overlap neither each other nor what it reads
bool any_overlap(Ranges outs) {
  for (const Range* o = outs.begin(); o != outs.end(); ++o)
    for (const Range* i = o + 1; i != outs.end(); ++i)
      if (overlaps(*o, *i)) return true;
  return false;
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
  const int64_t C = num_heads * 64;
  if (!ranks_fit(p, C)) return WKV7_ERR_SHAPE;
  if (!eps_ok(p.norm_time_eps) || !eps_ok(p.norm_channel_eps) || !eps_ok(p.group_norm_eps)) return WKV7_ERR_SHAPE;
  const int64_t row = C * 4, matrix = C * row;   // bytes
  const Ranges weights = {{p.norm_time_weight, row}, {p.norm_time_bias, row}, {p.norm_channel_weight, row},
                          {p.norm_channel_bias, row}, {p.mix[0], row}, {p.mix[1], row}, {p.mix[2], row},
                          {p.mix[3], row}, {p.mix[4], row}, {p.mix[5], row}, {p.receptance, matrix},
                          {p.key, matrix}, {p.value, matrix}, {p.output, matrix},
                          {p.decay_a, p.decay_rank * row}, {p.decay_b, p.decay_rank * row}, {p.decay_bias, row},
                          {p.rate_a, p.rate_rank * row}, {p.rate_b, p.rate_rank * row}, {p.rate_bias, row},
                          {p.gate_a, p.gate_rank * row}, {p.gate_b, p.gate_rank * row}, {p.key_removal, row},
                          {p.key_replacement, row}, {p.bonus, row}, {p.group_norm_weight, row},
                          {p.group_norm_bias, row}, {p.channel_mix, row}, {p.channel_key, 4 * matrix},
                          {p.channel_value, 4 * matrix}};
  if (int rc = check_pointers(weights)) return rc;
  const int64_t res = p.residual_a ? p.residual_rank * row : 0;
  const Ranges residual = {{p.residual_a, res}, {p.residual_b, res}, {p.residual_bias, row}};
  if (p.residual_a)
    if (int rc = check_pointers(residual)) return rc;
  if (rows == 0) return WKV7_OK;
  const int64_t shift = full_batch * row, elem = state_dtype == WKV7_DTYPE_BF16 ? 2 : 4;
  const int64_t needed = rwkv_decode::workspace_bytes(rows, num_heads);
  const Ranges outs = {{x, rows * row}, {state, full_batch * C * 64 * elem}, {shift_time_out, shift},
                       {shift_channel_out, shift}, {workspace, needed}};
  const Ranges shifts = {{shift_time_in, shift}, {shift_channel_in, shift}};
  if (int rc = check_pointers(outs)) return rc;
  if (int rc = check_pointers(shifts)) return rc;
  if (!batch_ids || (use_dither && !elapsed_t)) return WKV7_ERR_NULL_POINTER;
  if (!aligned(batch_ids, 4) || !aligned(elapsed_t, 4)) return WKV7_ERR_ALIGNMENT;
  if (workspace_bytes < needed) return WKV7_ERR_SHAPE;
  if (any_overlap(outs) || any_overlap(outs, shifts) || any_overlap(outs, weights) ||
      (p.residual_a && any_overlap(outs, residual)) ||
      any_overlap(outs, {{batch_ids, rows * 4}, {elapsed_t, full_batch * 4}}))
    return WKV7_ERR_OVERLAP;
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
  const int64_t C = num_heads * 64, needed = rwkv_decode::workspace_bytes(rows, num_heads);
  const Ranges weights = {{norm_weight, C * 4}, {norm_bias, C * 4}, {unembed, vocab * C * 4}};
  if (int rc = check_pointers(weights)) return rc;
  if (rows == 0) return WKV7_OK;
  const Ranges rows_in = {{x, rows * C * 4}}, outs = {{logits, rows * vocab * 2}, {workspace, needed}};
  if (int rc = check_pointers(rows_in)) return rc;
  if (int rc = check_pointers(outs)) return rc;
  if (workspace_bytes < needed) return WKV7_ERR_SHAPE;
  if (any_overlap(outs) || any_overlap(outs, weights) || any_overlap(outs, rows_in)) return WKV7_ERR_OVERLAP;
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
