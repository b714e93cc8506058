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
  int whole, lo, hi;                         // contexts of up to `whole` chunks (-1: none) are one slice; from 24 chunks on an eighth, lo to hi
};
// Below 256 pairs a context of 24 chunks and more has at most eight slices, up to slices of 8 chunks (shorter ones gain
// nothing: in threes 24 rows x 640 tokens 19.6 -> 20.4; 2 chunks in any case -> now, KV from HBM, Z
// for 8192 tokens, 8 kv heads, us: 8, 16, 24 rows x 1000 tokens 15.3 -> 14.2, 22.9 -> 21.7, 32.4 -> 27.4, a quarter of 24
// rows 1000 long and the others 100 27.0 -> 21.4); from 512 on one of 512 tokens is whole (10 chunks -> now: 64, 96 rows
// x 512 33.7 -> 31.8, 48.1 -> 44.4).  Longer slices are faster yet where the contexts are alike (8 chunks from 128 pairs on,
// 16 from 256, 32 from 512: 24 x 512 20.1 -> 18.7, 48 x 1000 47.8 -> 43.9, 64 x 1000 55.4 -> 53.5), but a row much longer
// than the others is then one wave for longer than the whole step takes: one of 500 tokens beside others of 64, 24, 31, 48,
// 63 rows 10.5 -> 12.4, 10.3 -> 13.1, 13.6 -> 16.2, 14.5 -> 16.8.  (Counting such rows in the kernels costs every
// step 0.5 us.)  fp8 chunks take twice the instructions: 64 pairs x 512 11.6, 12.8 in fours.  `fixed` > 0: for every launch.
inline DecodeLeast decode_least(int64_t pairs, bool kv_fp8, int fixed) {
  if (fixed > 0) return {-1, fixed < 2 ? 2 : fixed, fixed < 2 ? 2 : fixed};
  if (kv_fp8) return pairs >= DEC_LONG_PAIRS ? DecodeLeast{-1, 10, 10} : DecodeLeast{-1, 2, 2};
  if (pairs < DEC_LONG_PAIRS) return {-1, 2, 8};
  return {pairs >= 2 * DEC_LONG_PAIRS ? 16 : -1, 10, 10};
}
__host__ __device__ __forceinline__ int decode_min_chunks(const DecodeLeast& l, int nchunk) {
  const int e = nchunk < 24 ? 0 : (nchunk + 7) >> 3, p = e < l.lo ? l.lo : e < l.hi ? e : l.hi;
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
