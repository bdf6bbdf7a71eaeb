// Host build of althea_amd/csrc/irradiance_launch.hpp for
// tests/test_irradiance_launch.py.
#define __host__
#define __device__
#include "../../althea_amd/csrc/irradiance_launch.hpp"

using namespace althea;

extern "C" {
void grids(int size, int waves, unsigned* out) {
  const IrradianceGrid f = fold_blocks(size), t = texel_blocks(size, waves);
  out[0] = f.x, out[1] = f.y, out[2] = t.x, out[3] = t.y;
}
// Steps that a wave starting at step `wave` takes, `stride` apart, and the last of them.
long long fold_walk(int wave, int stride, int theta_steps, int polar_steps, int* last) {
  long long n = 0;
  for (FoldStep s = fold_advance({0, 0}, wave, theta_steps); s.polar < polar_steps;
       s = fold_advance(s, stride, theta_steps)) {
    if (s.polar < 0 || s.azimuth < 0 || s.azimuth >= theta_steps) return -1;
    last[0] = s.polar, last[1] = s.azimuth;
    ++n;
  }
  return n;
}
}
