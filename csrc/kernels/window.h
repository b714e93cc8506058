// Shared by the windowed attention kernels (attention_window.hip, window_prefill.hip, window_split.hip).
#pragma once
#include "common.h"
#include "launch.h"

namespace kgc {

// first position that a query at `pos` sees
__device__ __forceinline__ int first_visible(int pos, int window, bool chunked) {
  if (window <= 0) return 0;
  return chunked ? pos - pos % window : max(0, pos - window + 1);
}

// scaled score -> cap * tanh(score / cap) when a cap is set
__device__ __forceinline__ float cap_score(float s, float cap) {
  return cap > 0.f ? cap * tanhf(s / cap) : s;
}

// Of an element-wise output gate, the same for prompt and decode rows: e / (1 + e) or 1 / (1 + e) with e = 2^(-|x| log2 e),
// whose exponent loses its whole part in one rounding, and a reciprocal of 1 to 2 corrected once.  Units of 2^-24 from
// float64, rms and largest: gates of deviation 1 0.65 and 2.5, of 3 0.70 and 2.9, from -60 to 0 0.59 and 3.0.  1 /
// (1 + expf(-x)), whose subtractions -ffp-contract=fast fuses: 0.72 and 3.6, 1.09 and 11, 15.5 and 46, and twice the
// instructions; the hardware's reciprocal and 2^x alone 0.74 and 4.5, 1.17 and 12, 17.4 and 59.  In this
// order: capped prompts of 2 x 33 rows 12.4, 14.2 and 10.3 us, 64 x 100 33.6, 36.7 and 31.3.
__device__ __forceinline__ float gate_sigmoid(float x) {
  float a = fabsf(x);
  a = a > 110.f ? 110.f : a;                 // (e is zero from 104 on; NaN stays)
  const float n = __builtin_rintf(a * -1.44269502162933349609f);
  const float f = __builtin_fmaf(a, -1.925963033500e-8f, __builtin_fmaf(a, -1.44269502162933349609f, -n));
  const float e = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)n), d = 1.f + e;
  const float r = __builtin_amdgcn_rcpf(d);
  return (x < 0.f ? e : 1.f) * __builtin_fmaf(r, __builtin_fmaf(-d, r, 1.f), r);
}

// sigmoid of the element-wise output gate at (row t, column c of the concatenated heads)
template <typename T>
__device__ __forceinline__ float elem_gate(const WindowExtra& ex, int64_t t, int c) {
  if (ex.egate == nullptr) return 1.f;
  return gate_sigmoid(to_f(static_cast<const T*>(ex.egate)[t * ex.egs + c]));
}

}  // namespace kgc
