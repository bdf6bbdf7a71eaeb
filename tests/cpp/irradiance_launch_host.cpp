// Host build of althea_amd/csrc/irradiance_launch.hpp for
// tests/test_irradiance_launch.py.
#define __host__
#define __device__
#include "../../althea_amd/csrc/irradiance_launch.hpp"

using namespace althea;

extern "C" {
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
