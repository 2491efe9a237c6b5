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
// with the hardware exp2 and reciprocal (the network is trained with this
// same function and its derivative).  -z log2(e) = x (a x^2 + b).
constexpr float kGeluB = -2.302208198144325f;               // -2 sqrt(2/pi) log2(e)
constexpr float kGeluA = kGeluB * 0.044715f;
__device__ __forceinline__ float gelu_sigmoid(float x) {
  const float e = __builtin_amdgcn_exp2f(x * fmaf(kGeluA, x * x, kGeluB));
  return __builtin_amdgcn_rcpf(1.0f + e);
}
__device__ __forceinline__ float gelu(float x) { return x * gelu_sigmoid(x); }
__device__ __forceinline__ float gelu_grad(float x) {
  const float s = gelu_sigmoid(x);
  const float dz = 1.5957691216057308f * fmaf(3.0f * 0.044715f, x * x, 1.0f);
  return fmaf(x * s * (1.0f - s), dz, s);
}

}  // namespace hc
