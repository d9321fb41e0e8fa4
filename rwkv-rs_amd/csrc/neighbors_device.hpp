// Element-wise functions of the weight preparation's end
// (weight_prepare.rs:282-317), shared by the kernels that form it.
#pragma once

#include <hip/hip_runtime.h>

namespace rwkv_nb {

constexpr float kNormEps = 1e-12f;       // F.normalize's eps (weight_prepare.rs:313)
constexpr float kSoftplusLinear = 20.f;  // softplus(y) = y above this, as torch's

__device__ __forceinline__ float sigmoid1(float x) { return 1.f / (1.f + expf(-x)); }

__device__ __forceinline__ float softplus1(float y) {
  return y > kSoftplusLinear ? y : log1pf(expf(y));
}

}  // namespace rwkv_nb
