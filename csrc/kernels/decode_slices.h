// How K1w (attention_decode.hip) cuts contexts into z-slices of 32-token chunks; the decode kernel and its merge derive
// the same slices from these functions.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace kgc {

// From this many (sequence, kv head) pairs up the pairs by themselves fill the CUs
constexpr int DEC_LONG_PAIRS = 256;

// Chunks that a slice holds at least (2: the pipeline depth), a per-launch host choice: the graph's Z is sized for
// max_model_len, so at short contexts many-pairs grids would otherwise cut each context into slices of 2-3 chunks, each paying
// the q prologue and a partial write for little streaming.
struct DecodeLeast {
  int whole, lo, hi;                         // contexts of up to `whole` chunks (-1: none) are one slice; an eighth, from lo to hi
};
// Below 256 pairs a slice holds four chunks and a context has at most eight slices, up to slices of 8 chunks (slices of 2
// chunks, 3 from 17 on, 4 from 25 on -> now, 8 kv heads, calls with other KV each, from HBM, us: 8 rows x 600, 1000 tokens
// 20.2 -> 19.4, 24.2 -> 22.0; 16 x 400, 520, 740 18.7 -> 16.6, 21.9 -> 19.6, 24.1 -> 22.3; 24 x 400, 520, 640, 740 22.8 -> 20.9,
// 25.5 -> 23.4, 27.4 -> 25.7, 29.8 -> 29.0; 31 x 520 30.8 -> 28.4; one row of 500 beside others of 64, 16, 24, 31 rows
// 14.0 -> 13.3, 13.3 -> 12.9, 13.6 -> 13.9; 30 to 1000 tokens 16, 24 rows 23.0 -> 20.0, 26.8 -> 24.6; slices of 2 of any
// context: 24 x 1000 37.4 -> 32.2); from 512 on one of 512 tokens is whole (10 chunks -> now: 64, 96 rows
// x 512 33.7 -> 31.8, 48.1 -> 44.4).  Longer slices are faster yet where the contexts are alike (8 chunks from 128 pairs on,
// 16 from 256, 32 from 512: 24 x 520 23.4 -> 22.8, 48 x 1000 47.8 -> 43.9, 64 x 1000 55.4 -> 53.5), but a row much longer
// than the others is then one wave for longer than the whole step takes: one of 500 tokens beside others of 64, 24, 31, 48,
// 63 rows 12.9 -> 14.9, 13.9 -> 15.8, 13.6 -> 16.2, 14.5 -> 16.8.  (Counting such rows in the kernels costs every
// step 0.5 us.)  fp8 chunks take twice the instructions: 64 pairs x 512 11.6, 12.8 in fours.  `fixed` > 0: for every launch.
inline DecodeLeast decode_least(int64_t pairs, bool kv_fp8, int fixed) {
  if (fixed > 0) return {-1, fixed < 2 ? 2 : fixed, fixed < 2 ? 2 : fixed};
  if (kv_fp8) return pairs >= DEC_LONG_PAIRS ? DecodeLeast{-1, 10, 10} : DecodeLeast{-1, 2, 2};
  if (pairs < DEC_LONG_PAIRS) return {-1, 4, 8};
  return {pairs >= 2 * DEC_LONG_PAIRS ? 16 : -1, 10, 10};
}
__host__ __device__ __forceinline__ int decode_min_chunks(const DecodeLeast& l, int nchunk) {
  const int e = (nchunk + 7) >> 3, p = e < l.lo ? l.lo : e < l.hi ? e : l.hi;
  return nchunk <= l.whole ? l.whole : p;
}
// slices past the context are empty and the merge stops at decode_used_slices
__host__ __device__ __forceinline__ int decode_slice_chunks(int nchunk, int Z, int min_per) {
  const int per = (nchunk + Z - 1) / Z;
  return per < min_per ? min_per : per;
}
__host__ __device__ __forceinline__ int decode_used_slices(int nchunk, int Z, int min_per) {
  const int per = decode_slice_chunks(nchunk, Z, min_per);
  const int n = (nchunk + per - 1) / per;
  return n < Z ? n : Z;
}

}  // namespace kgc
