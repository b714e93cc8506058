// Shared by the windowed attention kernels (attention_window.hip, window_prefill.hip).
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

// Of an element-wise output gate, the same for prompt and decode rows.  The hardware's reciprocal and 2^x instead
// (64 x 100 prompt rows 31 us, so 37) are further off float64: gates of
// deviation 1, 3 and up to 10 by 0.75, 1.20 and 2.01 units of 2^-24 rms where this is by 0.73, 1.10 and 1.75.
__device__ __forceinline__ float gate_sigmoid(float x) { return 1.f / (1.f + expf(-x)); }

// sigmoid of the element-wise output gate at (row t, column c of the concatenated heads)
template <typename T>
__device__ __forceinline__ float elem_gate(const WindowExtra& ex, int64_t t, int c) {
  if (ex.egate == nullptr) return 1.f;
  return gate_sigmoid(to_f(static_cast<const T*>(ex.egate)[t * ex.egs + c]));
}

// column (lane & 15) of four rows of 16-bit elements in LDS: lanes 4 r .. 4 r + 3 of every 16 address
// row r, 4 elements each
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 ld_tr4(const void* p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                       (__attribute__((address_space(3))) s16x4*)p));
}

}  // namespace kgc
