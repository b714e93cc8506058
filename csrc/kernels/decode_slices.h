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
// the q prologue and a partial write for little streaming.  Where the least length would make two slices, the second one
// short, shorter ones are as fast or faster: `mid` for contexts of more than `from` and up to `to` chunks.
struct DecodeLeast {
  int per, from, to, mid;
};
// The pairs fill the chip the more the more there are, and a slice costs its q, its partial rows and their merge, so a context
// of up to that many chunks stays one.  With the KV from HBM, Z for 8192 tokens, us, with 2 chunks (10
// from 256 pairs on) -> now: 64 pairs x 300, 1000, 2000 tokens 10.5 -> 9.9, 14.6 -> 13.1, 22.9 -> 19.7; 128 x 128, 512,
// 1000 9.5 -> 8.9, 14.6 -> 14.0, 22.0 -> 19.4; 192 x 1000 29.3 -> 25.5; 256 x 512 19.4 -> 18.8; 512 x 512, 1000 32.8 -> 31.1,
// 55.7 -> 52.4.  fp8 chunks take twice the instructions, and are as they were: 64 x 512 11.6, 12.8 in fours.
// `fixed` > 0: for every launch.
inline DecodeLeast decode_least(int64_t pairs, bool kv_fp8, int fixed) {
  if (fixed > 0) return {fixed < 2 ? 2 : fixed, 0, 0, 0};
  if (kv_fp8) return {pairs >= DEC_LONG_PAIRS ? 10 : 2, 0, 0, 0};
  if (pairs >= 2 * DEC_LONG_PAIRS) return {32, 0, 0, 0};
  if (pairs >= DEC_LONG_PAIRS) return {16, 16, 24, 10};
  return pairs >= DEC_LONG_PAIRS / 2 ? DecodeLeast{8, 0, 0, 0} : DecodeLeast{4, 0, 8, 2};
}
__host__ __device__ __forceinline__ int decode_min_chunks(const DecodeLeast& l, int nchunk) {
  return nchunk > l.from && nchunk <= l.to ? l.mid : l.per;
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
