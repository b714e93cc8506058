// The items of the paged prompts' walk (attention_prefill.hip), and which of them a workgroup has.
#pragma once

#include <hip/hip_runtime.h>

namespace kgc {

constexpr int WALK_BLOCKS = 4;               // blocks of 32 rows in a work item of 128

// Item idx: 32-row block `block` of work item `work`, head group `group` of `groups`.  Neighbours are the head groups of the
// same rows: with a multiple of 8 of them an XCD sees one group in all rounds.  With fewer a work item's blocks change
// places by its number (the same for work and ~work, so that the mirrored round has them the other way): the last of short
// prompts have no rows, so that XCDs would be idle, and a workgroup's items of two rounds would both have rows or none.
// 8 heads on 1, two groups, 100, 200 x 64 rows: 17.3, 27.5 us -> 11.6, 19.5 (one-shot grid 12.0, 20.8).
__host__ __device__ inline void walk_item(int idx, int groups, int& work, int& block, int& group) {
  work = idx / (groups * WALK_BLOCKS);
  const int r = idx - work * (groups * WALK_BLOCKS);
  group = r % groups;
  block = WALK_BLOCKS - 1 - (r / groups ^ (groups % 8 == 0 ? 0 : (work ^ work >> 1) & (WALK_BLOCKS - 1)));
}

// The item of workgroup b of `grid` in round r: odd rounds run the other way, by eights (XCD by XCD) where an XCD has its group.
__host__ __device__ inline int walk_index(int r, int b, int grid, bool by_xcd) {
  const int turn = by_xcd && grid % 8 == 0 ? (grid - 8 - (b & ~7)) | (b & 7) : grid - 1 - b;
  return r * grid + (r & 1 ? turn : b);
}

}  // namespace kgc
