// Activations that are a launch of their own and the end of a projection too (gemm_prompt.hip): the same
// operations, so that both make the same bits of the same projection.
#pragma once
#include "common.h"

namespace kgc {

__device__ __forceinline__ float silu_mul_of(float g, float u) { return g / (1.f + __expf(-g)) * u; }

// xIELU: a x^2 + x / 2 above 0, b (e^x - 1 - x) + x / 2 below.  e^x - 1 - x without cancellation: the series
// x^2 (1/2 + x/6 + .. + x^6/40320) from -1/2 up, where its next term is 5e-8 of it, else 2^(x log2 e).
__device__ __forceinline__ float xielu_of(float x, float a, float b) {
  float p = 1.f / 40320.f;
  p = p * x + 1.f / 5040.f;
  p = p * x + 1.f / 720.f;
  p = p * x + 1.f / 120.f;
  p = p * x + 1.f / 24.f;
  p = p * x + 1.f / 6.f;
  p = p * x + 0.5f;
  const float e = x > -0.5f ? x * x * p : (__builtin_amdgcn_exp2f(x * 1.44269504088896340736f) - 1.f) - x;
  return x > 0.f ? a * x * x + 0.5f * x : b * e + 0.5f * x;
}

}  // namespace kgc
