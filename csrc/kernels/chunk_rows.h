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

// Whether prompt rows pay chunkwise, by what both ways take in us: token by token the states' way in and out and every
// row, by P H ceil(V / 64) units of 64 columns; chunkwise a chunk of each sequence whatever its rows, by P H ceil(V / 128)
// workgroups of the walk, of which a CU holds one, and P H of what goes before it.
//     t0 + tu units (+ t1 from 192 units on) + rows max(r0, ru units)   against   max(c0 + s0 wgs, c1 + cw wgs) + cp P H
// The constants are fitted to 3 to 12 rows of 1 to 512 sequences, rows the mean, which is at most the longest, and checked on
// equal lengths, where token by token loses least: 20 shapes of heads, 1 to 48 rows of 1 to 512 sequences that begin or go on
// from a state, each type.  What they choose, 2850 of 7350 steps, was at most 4 % slower (3 fp32 rows of GLA) and a third
// faster on average; what they leave was up to 1.4 times (mLSTM 1.5) as fast the other way, by more than 15 % in 290 steps.
// Measured, token by token -> chunkwise:
//                     1 x 8, 12, 24          8 x 8, 16        32 x 4, 6, 12            128 x 4, 8
//   GLA  8 x 256      12.4, 15.2, 26.6 -> 13.9   18.9, 25.7 -> 16.1   31.0, 34.7, 44.9 -> 30   89, 109 -> 69
//        2 x 128      11 rows 14.6 -> 13.2   12.4 -> 14.1     5 rows 12.0 -> 14.9      16.6 -> 21.8
//        4 x 64, 512  14.4, 14.6 -> 12.9, 13.8   12.4, 19.1 -> 13.9, 15.4   5 rows 11.9, 33.6 -> 15.2, 24.9   17, 89 -> 32, 64
//   delta 16 x 128    10.2, 12.8, 22.6 -> 19.9   15.0, 23.3 -> 21.7   21, 27, 38.7 -> 35       55, 81 -> 88
//        4 x 128, 32 x 128   22 rows 25.2, 21.2 -> 19.8   15.7, 25.6 -> 20.2, 24.3   12 rows 20, 63 -> 21.7, 53
//   mLSTM 4 of 256 x 512     25.2, 31.2 -> 19.0   27.1 -> 21.4   42, 49, 70 -> 42.6   151, 209 -> 139
//        8 of 128 x 128      17.3, 21.5 -> 12.5   6 rows 16.0 -> 13.2   16.5, 18.8 -> 15.9   41, 55 -> 47
//        16 of 128 x 64      15.3, 19.7 -> 12.3   6 rows 13.9 -> 13.1   14.5, 16.7 -> 24   39, 53 -> 79
struct ChunkCost { double t0, tu, t1, r0, ru, c0, s0, c1, cw, cp; int least; };
inline bool chunk_pays(const ChunkCost& k, long P, long Tp, long H, long V, double scale = 1.0) {
  if (P <= 0 || Tp < k.least * P) return false;
  const double units = (double)P * H * ((V + 63) / 64), wgs = (double)P * H * ((V + 127) / 128), rows = (double)Tp / P;
  const double slope = k.ru * units > k.r0 ? k.ru * units : k.r0, a = k.c0 + k.s0 * wgs, b = k.c1 + k.cw * wgs;
  return k.t0 + k.tu * units + (units > 192 ? k.t1 : 0) + rows * slope > scale * ((a > b ? a : b) + k.cp * P * H);
}

// By the rows alone, P sequences of Tp rows together: from `alone` rows of one sequence on, 24 in steps of 192, 16 in steps
// of 512 and 12 in steps of 1024.
inline bool chunk_rows_pay(long P, long Tp, long alone) {
  const long rows = Tp >= 1024 ? 12 : Tp >= 512 ? 16 : Tp >= 192 ? 24 : alone;
  return P > 0 && Tp >= (rows < alone ? rows : alone) * P;
}
// The same for the scans that prepare chunks in a workspace: by the rows, and by the costs in steps of fewer than
// 1024 rows (in larger ones short rows would start far more chunks than any other step, and the engine would set memory
// aside for their workspace).
inline bool chunk_rows_pay(const ChunkCost& k, long P, long Tp, long H, long V, long alone) {
  return chunk_rows_pay(P, Tp, alone) || (Tp < 1024 && chunk_pays(k, P, Tp, H, V));
}

// The delta rule's and GLA's, the costs as above.
inline bool delta_rows_pay(long P, long Tp, long H, long V) {
  constexpr ChunkCost COST{4.0, 0.0062, 0.0, 0.85, 0.0021, 21.5, 0.0, 15.5, 0.0468, 0.0, 8};
  return chunk_rows_pay(COST, P, Tp, H, V, 48);
}
inline bool gla_rows_pay(long P, long Tp, long H, long V) {
  constexpr ChunkCost COST{6.1, 0.0148, 2.0, 0.72, 0.0014, 13.6, 0.0247, 0.0, 0.0, 0.0147, 3};
  return chunk_rows_pay(COST, P, Tp, H, V, 32);
}

// Among steps of fewer than 1024 rows, at most `seqs` sequences of at most `len` rows and `rows` together, the one that
// goes chunkwise by `pay`(P, Tp) and has the largest workspace, of Tp / 32 + P chunks (P = 0: none does).  The costs
// say so neither at the fewest rows per sequence that they allow nor at the most sequences, so it is searched for.
struct ChunkStep { long P, Tp; };
template <typename F> inline ChunkStep most_chunks(F pay, long seqs, long rows, long len) {
  ChunkStep best{0, 0};
  if (rows > 1023) rows = 1023;
  for (long P = 1; P <= seqs && P <= rows; ++P)
    for (long Tp = rows < P * len ? rows : P * len; Tp >= P && Tp / 32 + P > best.Tp / 32 + best.P; --Tp)
      if (pay(P, Tp)) {
        best = {P, Tp};
        break;
      }
  return best;
}
inline ChunkStep delta_most_chunks(long H, long V, long seqs, long rows, long len) {
  return most_chunks([=](long P, long Tp) { return delta_rows_pay(P, Tp, H, V); }, seqs, rows, len);
}
inline ChunkStep gla_most_chunks(long H, long V, long seqs, long rows, long len) {
  return most_chunks([=](long P, long Tp) { return gla_rows_pay(P, Tp, H, V); }, seqs, rows, len);
}

// Tokens per segment, whole chunks of L and `least` of them at least, so that P sequences of Tp rows come to at most
// `want` segments
inline int segment_rows(int P, int Tp, int want, int L, int least) {
  const int seg = (Tp + want - P - 1) / (want - P);       // Tp / seg + P <= want
  const int rows = (seg + L - 1) / L * L;
  return rows < least * L ? least * L : rows;
}

}  // namespace kgc
