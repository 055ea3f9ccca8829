// zq3d_octree_plan.h -- the launches of the octree sweeps: which cell lists run side by side.
//
// A pass updates level 0 red, level 0 black, ..., level 3 black, each reading the newest pressures.
// Two lists of different levels whose leaves nowhere touch read nothing of each other, so their
// order is free: level 0 of the next pass may run beside level 2 of this one where no fine cell
// touches a 4^3 leaf, and so on.  Each list is put into the earliest launch after every earlier list
// of its own level and of every level that touches it; the pressures are those of the one-by-one
// order, bit for bit.  Leaves that step one level at a time (thresholds far enough apart) need four
// launches a pass instead of eight.  Plain C++ (compiled into tests on its own).
#pragma once

#include <stdint.h>

#include <algorithm>
#include <vector>

namespace zq3d {

constexpr int OCT_LISTS = 8;  // cell lists of the sweeps, 2 level + colour

// per launch the set of lists it updates (bit k: list k); counts: the lists' lengths (empty ones
// take no part); bit m of beside[L]: leaves of levels L and m touch
inline std::vector<uint8_t> oct_schedule(const uint32_t counts[OCT_LISTS], const uint32_t beside[4], int iters) {
    std::vector<uint8_t> plan;
    size_t done[4] = {0, 0, 0, 0};  // launches up to the newest list of each level
    for (int it = 0; it < iters; it++)
        for (int k = 0; k < OCT_LISTS; k++) {
            if (!counts[k]) continue;
            const int L = k / 2;
            size_t at = done[L];
            for (int m = 0; m < 4; m++)
                if (beside[L] >> m & 1) at = std::max(at, done[m]);
            if (plan.size() <= at) plan.resize(at + 1, 0);
            plan[at] |= (uint8_t)(1u << k);
            done[L] = at + 1;
        }
    return plan;
}

}  // namespace zq3d
