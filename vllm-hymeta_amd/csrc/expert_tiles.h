// Tiles of a grouped expert product of few slots an expert: what a workgroup of one column of tiles x some slots works on.
#pragma once

#include "act_types.h"

#include <algorithm>

namespace hymeta {
namespace {

constexpr int kExpertDies = 8;

// Slots [row, row + rows) of expert e, column `col`.
struct ExpertTile { int e, row, rows, col; };

// An expert's slots are cut into as few equal tiles of up to tile_rows as hold them, which stand next to each other in a column, column
// behind column; a die takes an eighth of all tiles in a row (block = die + 8 (tile of the die)), so that weights and an expert's
// slots are read from its L2.  A lane looks after an expert.  Wave-uniform; false: nothing to do.
__device__ __forceinline__ bool expert_tile(const int32_t* offsets, int begin, int end, int cols, int tile_rows, ExpertTile* p) {
  const int lane = threadIdx.x & 63;
  int lo = 0, hi = 0;
  auto tiles_of = [&](int e0) {
    const int e = min(e0 + lane, end - 1);
    lo = offsets[e], hi = offsets[e + 1];
    return e0 + lane < end ? (hi - lo + tile_rows - 1) / tile_rows * cols : 0;
  };
  int total = 0;
  for (int e0 = begin; e0 < end; e0 += 64) total += __builtin_amdgcn_readlane(lane_sums(tiles_of(e0)), 63);
  const int64_t all = total;
  const int die = blockIdx.x % kExpertDies, first = static_cast<int>(all * die / kExpertDies), count = static_cast<int>(all * (die + 1) / kExpertDies) - first;
  int t = blockIdx.x / kExpertDies;
  if (t >= count) return false;
  t += first;
  for (int e0 = begin; e0 < end; e0 += 64) {
    const int mine = tiles_of(e0), upto = lane_sums(mine);
    const uint64_t past = __ballot(t < upto);
    if (past == 0) {
      t -= __builtin_amdgcn_readlane(upto, 63);
      continue;
    }
    const int at = __builtin_ctzll(past);
    t -= __builtin_amdgcn_readlane(upto - mine, at);
    lo = __builtin_amdgcn_readlane(lo, at), hi = __builtin_amdgcn_readlane(hi, at);
    const int row_tiles = __builtin_amdgcn_readfirstlane((hi - lo + tile_rows - 1) / tile_rows), col = __builtin_amdgcn_readfirstlane(t / row_tiles);
    const int each = __builtin_amdgcn_readfirstlane((hi - lo + row_tiles - 1) / row_tiles);
    p->e = e0 + at, p->col = col, p->row = lo + (t - col * row_tiles) * each, p->rows = min(each, hi - p->row);
    return true;
  }
  return false;
}

// Slots of a tile at most: fewer than `most` where the tiles then still run all at once (an expert may have a fifth more than the average).
// 2 experts of 4096 x 4096 and 40 rows in bf16 142 -> 106 us.
inline int expert_tile_rows(int most, int64_t max_rows, int experts, int cols) {
  const int64_t likely = (max_rows + max_rows / 5 + experts - 1) / experts;
  auto at_once = [&](int rows) { return (likely + rows - 1) / rows * experts * cols <= 256; };
  return at_once(64) ? 64 : at_once(128) ? 128 : most;
}

// The host knows the slots, not how the experts share them.
inline unsigned expert_tile_grid(int64_t max_rows, int experts, int cols, int tile_rows) {
  const int64_t tiles = cols * ((max_rows + tile_rows - 1) / tile_rows + experts);
  return static_cast<unsigned>((tiles + kExpertDies - 1) / kExpertDies * kExpertDies);
}

}  // namespace
}  // namespace hymeta
