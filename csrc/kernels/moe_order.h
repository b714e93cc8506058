// Which order the blocks of K14m's 1-D grid have (gemm_decode.hip).
#pragma once

namespace kgc {

// Row blocks fastest: a column tile's blocks (one expert each) are dispatched together, so each XCD's L2 holds the
// activation rows of the experts it is dealt -- or column tiles fastest (true), each block's over all XCDs.  us a call with
// the weights not in the caches, row blocks fastest -> column tiles fastest:
//   few pairs, most blocks without rows: with 8 or 16 blocks to a column tile the ones that have rows were
//     all on one XCD each.  8 experts of 4096 x 14336, top 2, 1 and 2 rows 266 -> 128, 318 -> 238; 16 of 4096 x 6400
//     1, 4 rows 213 -> 81, 281 -> 200;
//   the down projection of 64-row blocks that all have rows (its K slices already go over the XCDs, its blocks then
//     did not), and of few experts at any rows: 8 experts 8 to 64 rows, both projections, 540 -> 485, 16 experts 32 to 256 rows
//     505 -> 440 (gate_up so: 2 % slower); 4 of 4096 x 14336 2, 4, 32, 64 rows 67 -> 65, 101 -> 73, 117 -> 78, 115 -> 104.  Not
//     where a block has few tiles (12 experts of 2048 x 5504 128 rows 50 -> 54, 3 of 2048 x 8192 8 rows 20 -> 21), nor
//     blocks of more than 16 experts, which are on all XCDs anyway: 32 of 2048 x 1408 64, 256 rows 35.5 -> 37.4, 33.3 -> 38.4;
//   gate_up of few experts of 64-row blocks where all its tiles are one round of workgroups: 4 of 2048 x 8192 3, 8, 64
//     rows 50 -> 40, 63 -> 45, 64 -> 44, 2 of 4096 x 14336 8 rows 86 -> 74; with more tiles, 4 of 4096 x 14336, 2, 4, 32 rows 123 -> 137,
//     146 -> 154, 153 -> 162;
//   gate_up of 128-row blocks, a multiple of 8, in many column tiles: 8 experts 512, 1024 rows 851 -> 753, 1475 -> 1388
//     (28 tiles to a block: 224 -> 236; more blocks to an expert would each stream its weights).
// Between, row blocks: 8 experts 4 to 6 rows 364 -> 378, 128 to 384 rows 509 -> 525 and more; 64 experts 8 rows 115 -> 130.
// (gate_up of 128-row blocks that are no multiple of 8 is not pinned, and 4 to 8 % slower than by column tiles: 8 experts 520,
// 600, 760, 960 rows 817 -> 785, 1247 -> 1177, 1211 -> 1152, 1381 -> 1272.)
inline bool moe_columns_first(bool gate_up, int experts, int block_rows, int blocks, int tiles, int pairs) {
  if (pairs < (experts < 16 ? experts : 16)) return true;
  if (!gate_up) return block_rows == 64 && tiles >= 16 && experts <= 16 && (experts <= 4 || pairs >= 2 * experts);
  return (block_rows == 64 && experts <= 4 && experts * tiles <= 256) ||
         (block_rows == 128 && blocks % 8 == 0 && blocks <= 3 * experts && tiles >= 48);
}

}  // namespace kgc
