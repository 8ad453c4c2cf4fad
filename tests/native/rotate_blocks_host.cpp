// Host build of the rotating launches' grid (chaoslibrary_amd/csrc/
// rotate_plan.hpp), for tests/test_rotate_blocks_cpu.py.
#include "rotate_plan.hpp"

extern "C" unsigned blocks_host(long long cus, int waves, int block) { return chaos::rotate_blocks(cus, waves, block); }
