// Shared by the surrogate network's forward and backward kernels.
#pragma once

#include "hc_common.h"

namespace hc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(__bf16 v) { return (float)v; }
__device__ __forceinline__ __bf16 f2bf(float v) { return (__bf16)v; }  // RNE

// GELU in its tanh form (torch.nn.GELU(approximate="tanh")):
// 0.5 x (1 + tanh(z / 2)) = x * sigmoid(z), z = 2 sqrt(2/pi) (x + 0.044715 x^3),
// with the hardware exp and reciprocal (the network is trained with this
// same function and its derivative).
__device__ __forceinline__ float gelu_z(float x) {
  return 1.5957691216057308f * fmaf(0.044715f * x, x * x, x);
}
__device__ __forceinline__ float gelu(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __expf(-gelu_z(x)));
}
__device__ __forceinline__ float gelu_grad(float x) {
  const float s = __builtin_amdgcn_rcpf(1.0f + __expf(-gelu_z(x)));
  const float dz = 1.5957691216057308f * fmaf(3.0f * 0.044715f, x * x, 1.0f);
  return fmaf(x * s * (1.0f - s), dz, s);
}

}  // namespace hc
