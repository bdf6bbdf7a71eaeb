// Host build of althea_amd/csrc/batch_launch.hpp for tests/test_batch_launch.py.
#include "../../althea_amd/csrc/batch_launch.hpp"

extern "C" int blocks_of(int cus, int waves_per_cu, int block_waves) {
  return althea::batch_blocks(cus, waves_per_cu, block_waves);
}
