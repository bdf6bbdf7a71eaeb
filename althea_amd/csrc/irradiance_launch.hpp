// Grids and step arithmetic of the irradiance kernels, host and device.
#pragma once

namespace althea {

// Grids in two dimensions: HIP takes less than 2^32 threads along x, which the
// blocks of a cube of 2 365 (1 024 threads an orbit) or 3 345 (64 a texel) in
// one row of blocks pass.
struct IrradianceGrid {
  unsigned x, y;
};

// A block per orbit of eight texels: x = cv, y = axis * half + cu.
__host__ inline IrradianceGrid fold_blocks(int size) {
  const unsigned half = (static_cast<unsigned>(size) + 1) / 2;
  return {half, 3 * half};
}

// A wave per texel: x = blocks of `waves` texels of a face, y = the face.
__host__ inline IrradianceGrid texel_blocks(int size, int waves) {
  return {(static_cast<unsigned>(size) * static_cast<unsigned>(size) + waves - 1) / waves, 6};
}

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
