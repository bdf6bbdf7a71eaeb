// Step arithmetic of the folded irradiance kernel, host and device.
#pragma once

namespace althea {

// A step of an orbit: the patch of 8 polar rows 8 polar.. by 8 azimuths
// 8 azimuth...  Step numbers are never formed: theta_steps x polar groups passes
// 2^31 for sample counts that the entry points accept (8 x 128 source, 100 000
// azimuths: 2.5e9 steps).
struct FoldStep {
  int polar, azimuth;
};

// `stride` steps after `s`, the azimuth groups running first.
__host__ __device__ inline FoldStep fold_advance(FoldStep s, int stride, int theta_steps) {
  s.azimuth += stride;
  if (s.azimuth >= theta_steps) {
    const int rows = s.azimuth / theta_steps;
    s.polar += rows;
    s.azimuth -= rows * theta_steps;
  }
  return s;
}

}  // namespace althea
