// Blocks and query ranges of the point prefilter, host and device.
#pragma once

#include <stddef.h>

namespace althea {

// Blocks of `waves` waves for `count` queries, one a wave, at most `most`.
__host__ inline int point_blocks(int count, int waves, int most) {
  const int blocks = (count - 1) / waves + 1;
  return blocks < most ? blocks : most;
}

// The queries of a wave: `first` and every `stride` after it, below the count.
// 64-bit: near 2^31 queries the walk steps past what an int holds.
struct PointWalk {
  size_t first, stride;
};
__host__ __device__ inline PointWalk point_walk(unsigned block, unsigned blocks, unsigned wave, unsigned waves) {
  return {static_cast<size_t>(block) * waves + wave, static_cast<size_t>(blocks) * waves};
}

}  // namespace althea
