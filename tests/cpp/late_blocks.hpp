// Forced into the traversal kernels of bin/libsepgraph_late.so (see Makefile):
// blocks outside the team read every round's counters 100 us late, so that
// whatever a team phase changes under them is changed before they read.
#pragma once

#include "frontier.hpp"

namespace sg {

__device__ __forceinline__ void read_counts_late(const FrontierCtr *c, unsigned long long *s_lvl)
{
    // other XCDs' blocks, and most of the lowest one's that are not members
    if (threadIdx.x < kWave && (xcc_id() != 0 || blockIdx.x >= 10 * kTeamMax)) {
        const long long t0 = wall_clock64();
        while (wall_clock64() - t0 < 10000) __builtin_amdgcn_s_sleep(8);  // 100 MHz
    }
    read_counts(c, s_lvl);
}

}  // namespace sg

#define read_counts read_counts_late
