// The exact GELU and its derivative as every kernel of this library evaluates them, so
// that an activation fused into a GEMM's output tiles gives the bits of the activation
// kernel behind it.
#pragma once
#include <math.h>

#include <type_traits>

#include "common.h"

namespace fmoe {

// gelu(x) = x Phi(x), gelu'(x) = Phi(x) + x phi(x); Phi through erfc so that the
// negative tail keeps its relative accuracy.
__device__ __forceinline__ double gelu_f64(double x) { return 0.5 * x * erfc(-x * M_SQRT1_2); }
__device__ __forceinline__ double gelu_grad_f64(double x) {
  return 0.5 * erfc(-x * M_SQRT1_2) + x * exp(-0.5 * x * x) * 0.3989422804014327;
}

__device__ __forceinline__ float gelu_direct(float x) {
  return 0.5f * x * (1.f + erff(x * 0.70710678118654752f));
}
__device__ __forceinline__ double gelu_direct(double x) { return gelu_f64(x); }
__device__ __forceinline__ float gelu_grad_direct(float x) {
  return 0.5f * (1.f + erff(x * 0.70710678118654752f)) +
         x * expf(-0.5f * x * x) * 0.3989422804014327f;
}
__device__ __forceinline__ double gelu_grad_direct(double x) { return gelu_grad_f64(x); }

// ReLU of 16-bit patterns; whether a negative value is a NaN only its bits above infinity's
// tell.  A NaN stays one in both directions, and the gradient of an inactive unit is zero
// whatever arrives there (infinities and NaNs too), as in torch.
template <typename T> constexpr uint16_t kInf16 = std::is_same<T, __half>::value ? 0x7c00 : 0x7f80;
template <typename T>
__device__ __forceinline__ uint16_t relu_fwd16(uint16_t v) {
  return (v & 0x8000u) && (v & 0x7fffu) <= kInf16<T> ? 0 : v;
}
template <typename T>
__device__ __forceinline__ uint16_t relu_bwd16(uint16_t d, uint16_t pre) {
  return pre == 0 || ((pre & 0x8000u) && (pre & 0x7fffu) <= kInf16<T>) ? 0 : d;
}
// two values to a word
template <typename T>
__device__ __forceinline__ uint32_t relu_fwd_pair(uint32_t v) {
  return relu_fwd16<T>((uint16_t)v) | ((uint32_t)relu_fwd16<T>((uint16_t)(v >> 16)) << 16);
}
template <typename T>
__device__ __forceinline__ uint32_t relu_bwd_pair(uint32_t d, uint32_t pre) {
  return relu_bwd16<T>((uint16_t)d, (uint16_t)pre) |
         ((uint32_t)relu_bwd16<T>((uint16_t)(d >> 16), (uint16_t)(pre >> 16)) << 16);
}

}  // namespace fmoe
