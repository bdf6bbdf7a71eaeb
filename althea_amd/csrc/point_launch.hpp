// Blocks and query ranges of the point prefilter, host and device.
#pragma once

#include <stddef.h>

namespace althea {

// Blocks of `waves` waves for `count` queries, `per` a wave, at most `most`.
__host__ inline int point_blocks(int count, int waves, int per, int most) {
  const int blocks = (count - 1) / (waves * per) + 1;
  return blocks < most ? blocks : most;
}

// Lanes of a query: 64, or 16, 4 or 1 where a query has few samples and there are
// queries enough to fill the GPU all the same.  A wave pays a query's frame and
// the sums across its lanes whatever the samples (2^20 queries: 480 us with 64
// lanes from 1 sample to 64), and the last step's idle lanes; a lane that walks
// more samples alone waits longer, which shows where the queries are few.  Each
// step down asks for fewer than 16 samples a lane and as many queries as make up
// for that wait, by the steps a lane then walks.  1024 x 512 source, us a call
// with 64, 16, 4 and 1 lanes:
//   8 192 queries, 64 samples   10.2 10.0 18.8 53.6    128: 11.9 13.3 32 107
//   16 384, 128                 17.3 16.5 32 107       255: 23.6 26.7 62 225
//   32 768, 16                  22.0 10.3 10.4 17.8    255: 41.8 39.9 62 225
//   65 536, 32                  37.3 17.7 16.3 29.0     64: 37.5 24.5 25.4 53.6
//   131 072, 4                  68.8 23.0 10.6 10.4     8: 68.8 22.9 12.2 12.5
//   2^20, 15                    510 139 82 66          128: 738 539 569 550
__host__ inline int point_lanes(int samples, int count) {
  int lanes = 64;
  while (lanes > 1) {
    const int next = lanes / 4, steps = (samples + next - 1) / next;
    if (steps > 16 || static_cast<long long>(count) * next < 32768ll * steps) break;
    lanes = next;
  }
  return lanes;
}

// Whether the coarse levels go through LDS: not for a lane's one to three
// samples (2^20 queries of 1 sample: 18.3 us staged, 14.0 from memory; of 2, 20.9
// and 18.0; of 8, 41 and 44).
__host__ inline bool point_stages(int samples, int lanes) { return lanes > 1 || samples > 3; }

// The queries of a wave: `per` from `first` and from every `stride` after it,
// below the count.  64-bit: near 2^31 queries the walk steps past what an int holds.
struct PointWalk {
  size_t first, stride;
};
__host__ __device__ inline PointWalk point_walk(unsigned block, unsigned blocks, unsigned wave, unsigned waves,
                                                unsigned per) {
  return {(static_cast<size_t>(block) * waves + wave) * per, static_cast<size_t>(blocks) * waves * per};
}

}  // namespace althea
