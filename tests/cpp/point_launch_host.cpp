// Host build of althea_amd/csrc/point_launch.hpp for tests/test_point_launch.py.
#define __host__
#define __device__
#include "../../althea_amd/csrc/point_launch.hpp"

using namespace althea;

extern "C" {
int lanes_of(int samples, int count) { return point_lanes(samples, count); }

// Queries that the waves of a launch take in all, and the largest; -1 where a
// walk does not end below the count.
long long point_total(int count, int waves, int per, int most, long long* largest) {
  const int blocks = point_blocks(count, waves, per, most);
  long long total = 0;
  *largest = -1;
  for (int b = 0; b < blocks; ++b)
    for (int w = 0; w < waves; ++w) {
      const PointWalk k = point_walk(b, blocks, w, waves, per);
      if (k.first >= static_cast<size_t>(count)) continue;
      const size_t n = (static_cast<size_t>(count) - 1 - k.first) / k.stride + 1;
      size_t q = k.first;
      for (size_t i = n > 3 ? n - 3 : 0; i < n; ++i) q = k.first + i * k.stride;
      const size_t next = q + k.stride;
      if (next < q || next < static_cast<size_t>(count)) return -1;
      const size_t here = static_cast<size_t>(count) - q < static_cast<size_t>(per) ? count - q : per;
      if (static_cast<long long>(q + here) - 1 > *largest) *largest = static_cast<long long>(q + here) - 1;
      total += static_cast<long long>((n - 1) * per + here);
    }
  return total;
}
}
