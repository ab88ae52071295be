// Launch sizes that follow from the sizes of a simulation (plain C++, so that host tests can read them too).
#pragma once
#include <algorithm>

namespace lsd {

// Blocks of 1024 threads of the single-launch broad phase, which must all be on the GPU together: one per 512
// particles or per 16,384 search cells (the cell loops of a sparse domain, such as an ensemble of drums far apart),
// at least 8, at most one per CU (a block takes a CU's registers).  So 32 simulations of up to 4,096 particles, or six
// of 20,000, can be stepped at once from threads or processes without one's barriers waiting for another's blocks.
// A wider grid makes one simulation's rebuild faster (passes of 4,000 bodies in a quarter sector 5 % with 63 blocks for
// 8, of 20,000 falling 2 % with 64 for 40) and is the caller's choice (broad_phase_blocks): as the rule, one block per 64
// particles left room for four simulations of 4,000, and a fifth waited until its barrier gave up.
inline int broadPhaseBlocks(long long particles, long long cells, int numCU) {
  return int(std::min<long long>(numCU, std::max<long long>({8, (particles + 511) / 512, (cells + 16383) / 16384})));
}

}  // namespace lsd
