// Launch sizes that follow from the sizes of a simulation, and how a launch shares its work (plain C++ for the host, so
// that host tests can run them too).
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

// The candidate search gives each master 32 lanes of a block.  As separate launches, blocks of 256 threads: 8 masters at
// a time, as many blocks as give each group one.
constexpr int kFindLanes = 32, kFindThreads = 256;
inline int pairsFindBlocks(long long particles) {
  constexpr int kGroups = kFindThreads / kFindLanes;
  return int(std::max<long long>(1, (particles + kGroups - 1) / kGroups));
}

#ifdef __HIPCC__
#define LSD_RULE __host__ __device__
#else
#define LSD_RULE
#endif
// The masters of a block of GROUPS groups: its share of the sorted order, GROUPS consecutive ones at a time (a turn of the
// block) from all over it (consecutive ones meet the same cells; sizes may be sorted in space, so no block gets one
// end).
template <int GROUPS>
struct MasterShare {
  int blocks, block;
  int chunk;  // masters of a full share
  LSD_RULE MasterShare(int nP, int blocks_, int block_) : blocks(blocks_), block(block_) {
    chunk = (nP + blocks * GROUPS - 1) / (blocks * GROUPS) * GROUPS;
  }
  LSD_RULE int at(int i) const {  // sorted position of the block's i-th master (may be >= nP)
    return (i / GROUPS * blocks + block) * GROUPS + i % GROUPS;
  }
};
#undef LSD_RULE

}  // namespace lsd
