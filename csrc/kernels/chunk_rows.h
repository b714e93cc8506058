// Host side: whether prompt rows are worth a chunkwise scan that prepares whole chunks of 32 tokens, and
// whether it can address them.
#pragma once

namespace kgc {

// The walks hold offsets inside a chunk (64 rows of `stride` elements, some as 24-bit products) and inside
// a head's state (256 rows of at most `cols` columns, all heads' together) in 32 bits, and put `blocks`
// workgroups on a grid's second axis.  Larger calls stay token by token, where offsets have 64 bits.
inline bool chunk_fits(long stride, long cols, long blocks) {
  return stride < (1 << 22) && cols < 1000000 && blocks <= 65535;
}

// P sequences of Tp rows together; `alone`: rows from which one sequence by itself pays.  Token by token
// a step costs its longest sequence and, once the chip is full, its rows; chunkwise it costs its chunks,
// one at least per sequence, full or not.  Token by token -> chunkwise in us, 16 heads of 128 x 128 (delta
// rule) and 8 of 128 x 256 (GLA):
//                        delta           GLA
//   1 x 24, 32, 44       22.5 -> 27.6, 27.7 -> 27.9, 36.8 -> 33.6;  26.5 -> 31.2, 31.8 -> 31.7, 43.1 -> 36.2
//   4 x 24, 40           22.8 -> 28.5, 35.2 -> 37.7;  28.2 -> 32.7, 42.8 -> 39.8
//   8 x 16, 24           23.8 -> 30.5, 35.4 -> 33.1;  25.7 -> 34.5, 37.2 -> 36.5
//   32 x 12, 16          43.1 -> 47.7, 51.9 -> 48.0;  48.7 -> 50.7, 56.1 -> 52.8
//   512 x 7, 128 x 12    386 -> 449, 152 -> 133;      509 -> 550, 173 -> 153
//   1024 x 1             473 -> 880;                  639 -> 1044
inline bool chunk_rows_pay(long P, long Tp, long alone) {
  const long rows = Tp >= 1024 ? 12 : Tp >= 512 ? 16 : Tp >= 192 ? 24 : alone;
  return P > 0 && Tp >= (rows < alone ? rows : alone) * P;
}

// Tokens per segment, whole chunks of L and `least` of them at least, so that P sequences of Tp rows come to at most
// `want` segments
inline int segment_rows(int P, int Tp, int want, int L, int least) {
  const int seg = (Tp + want - P - 1) / (want - P);       // Tp / seg + P <= want
  const int rows = (seg + L - 1) / L * L;
  return rows < least * L ? least * L : rows;
}

}  // namespace kgc
