// The exact GELU and its derivative as every kernel of this library evaluates them, so
// that an activation fused into a GEMM's output tiles gives the bits of the activation
// kernel behind it.
#pragma once
#include <math.h>

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

}  // namespace fmoe
