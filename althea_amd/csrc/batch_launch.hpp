// Grid of the persistent batched prefilter.
#pragma once

namespace althea {

// Blocks of `block_waves` waves for `waves_per_cu` waves a CU, one a CU at least:
// settings of 4 to 7 waves in blocks of 8 would leave half to an eighth of the
// CUs without work (12 maps of 1024, 512 and 256 at 4 waves: 4.86 ms, 2.46 with a
// block on every CU; blocks of 4 waves at 4, which an earlier setting was chosen
// for, 5.67).
inline int batch_blocks(int cus, int waves_per_cu, int block_waves) {
  const int blocks = cus * waves_per_cu / block_waves;
  return blocks > cus ? blocks : cus;
}

}  // namespace althea
