// Launchers of the decode step's kernels (decode.hip); the C ABI
// (decode_api.cpp) checks every argument before it calls them.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/rwkv_decode.h"

namespace rwkv_decode {

typedef uint16_t bf16_t;

struct CellCall {
  const rwkv_decode_cell_params* p;
  float* x;
  const int32_t* batch_ids;
  void* state;
  const float *shift_time_in, *shift_channel_in;
  float *shift_time_out, *shift_channel_out;
  const int32_t* elapsed_t;
  int rows, H, full_batch;
  bool state_bf16;
  int use_dither;
  void* workspace;
};
struct HeadCall {
  const float *x, *norm_weight, *norm_bias, *unembed;
  float eps;
  int rows, H;
  int64_t vocab;
  bf16_t* logits;
  void* workspace;
};

// bf16 elements per row of the workspace, in multiples of C (decode.hip lays them out)
constexpr int64_t kWorkspaceRows = 14;
inline int64_t workspace_bytes(int64_t rows, int64_t H) { return kWorkspaceRows * rows * H * 64 * 2; }

hipError_t launch_cell(const CellCall& c, hipStream_t stream);
hipError_t launch_head(const HeadCall& c, hipStream_t stream);

}  // namespace rwkv_decode
