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

// Rows per sequence from which P sequences of Tp rows together pay chunkwise: `rows` for fewer than 8 sequences, than 32,
// than 128, and more.  Token by token a step costs its longest sequence and, once the chip is full, its rows;
// chunkwise it costs its chunks, one at least per sequence, full or not.  From 1024 rows on 12 in any case: below, so
// short rows would start more chunks than the engine's memory profile has.  Token by token -> chunkwise in
// us, 16 heads of 128 x 128 (delta rule) and 8 of 128 x 256 (GLA), the shortest sequence three quarters of the longest:
//                          delta                                      GLA
//   1 x 16, 20, 24         16.0 -> 20.0, 19.8 -> 20.0, 22.5 -> 19.9;  17.9 -> 13.9, 24.0 -> 14.0, 26.6 -> 13.9
//   1 x 8, 12              10.3 -> 19.9, 13.1 -> 19.9;                12.4 -> 13.9, 15.2 -> 13.9
//   4 x 12, 16, 24         13.5 -> 20.8, 16.6 -> 20.8, 22.8 -> 20.7;  16.8 -> 15.4, 20.3 -> 15.4, 28.8 -> 15.3
//   8 x 8, 12, 16          15.0 -> 21.6, 19.4 -> 21.7, 23.4 -> 21.8;  18.9 -> 16.1, 22.2 -> 16.0, 25.7 -> 16.2
//   16 x 6, 8, 16          14.8 -> 23.7, 16.9 -> 24.1, 25.2 -> 24.2;  18.3 -> 18.4, 20.4 -> 18.7, 28.4 -> 18.8
//   32 x 4, 8, 12          21.1 -> 35.7, 30.6 -> 35.5, 38.8 -> 35.3;  31.0 -> 30.2, 38.3 -> 30.0, 44.9 -> 29.6
//   128 x 4, 8, 12         54.9 -> 89.2, 81.5 -> 86.8, 112 -> 88.7;   89.3 -> 69.0, 109 -> 66.4, 135 -> 68.4
//   300 x 3, 512 x 7, 12   -, 329 -> 341, 471 -> 355;                 191 -> 173, 415 -> 294, 522 -> 303
inline bool chunk_rows_pay(long P, long Tp, const int (&rows)[4]) {
  return P > 0 && Tp >= P * (Tp >= 1024 ? 12 : rows[P < 8 ? 0 : P < 32 ? 1 : P < 128 ? 2 : 3]);
}

// Tokens per segment, whole chunks of L and `least` of them at least, so that P sequences of Tp rows come to at most
// `want` segments
inline int segment_rows(int P, int Tp, int want, int L, int least) {
  const int seg = (Tp + want - P - 1) / (want - P);       // Tp / seg + P <= want
  const int rows = (seg + L - 1) / L * L;
  return rows < least * L ? least * L : rows;
}

}  // namespace kgc
