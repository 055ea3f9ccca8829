// zq3d_ens_plan.h -- how long a launch of the ensemble's register sweeps is predicted to take, from how its
// tiles fill the CUs: plain C++ that the launcher and a host test share.
#pragma once

#include <algorithm>
#include <vector>

#include "zq3d_quad_cut.h"

namespace zq3d {

// Steps of chunk bz's tiles: the chunk's planes and the pipeline's fill.
inline int ens_chunk_steps(const QuadCut& c, int K, int bz, int D) {
    return quad_z_begin(c, K, bz + 1, D) - quad_z_begin(c, K, bz, D) + (bz ? 4 * K - 2 : 2 * K - 1);
}
// Predicted microseconds of a tile.
inline double ens_tile_us(int steps, int K, int cx, int nw) { return 1.5 + steps * quad_step_us(K, cx, nw); }

// n tiles of the same predicted time
struct EnsRun {
    double us;
    long long n;
};

// When the last of the runs' tiles ends if they start in this order (longest first), XCD b % 8 takes block b,
// and each of an XCD's 32 CUs takes its next tile when it has finished one.  XCD 0 is the last to end:
// its i-th tile is as long as any other's i-th, and it has as many.  A tile goes to the CU that is free
// first; the CUs' free times stay sorted in two queues, those from before the run and those that a tile
// of the run set, and whole rounds of a run are added at once, so a run of any length costs a few dozen
// steps.  (One by one with a heap, and with every shape's tables made at once, creating 512 members of
// 64^3 took 20 ms and two of 512^3 44; now 2.3 and 2.7.)
inline double ens_fill_us(const std::vector<EnsRun>& runs) {
    constexpr int CUS = 32;
    double cu[CUS] = {}, set[CUS], merged[CUS];
    long long at = 0;
    for (const EnsRun& r : runs) {
        long long m = (at + r.n + 7) / 8 - (at + 7) / 8;
        at += r.n;
        int old = 0, head = 0, tail = 0;
        auto one = [&] {
            const bool fresh = old == CUS || (head < tail && set[head % CUS] < cu[old]);
            const double t = (fresh ? set[head++ % CUS] : cu[old++]) + r.us;
            set[tail++ % CUS] = t;
        };
        while (m > 0 && old < CUS) one(), m--;
        if (m > 0) {  // every free time is this run's: in order, and within one tile of each other
            const long long rounds = m / CUS;
            for (double& t : set) t += (double)rounds * r.us;
            for (m -= rounds * CUS; m > 0; m--) one();
        }
        int n = 0;
        while (old < CUS || head < tail)
            merged[n++] = old == CUS || (head < tail && set[head % CUS] < cu[old]) ? set[head++ % CUS] : cu[old++];
        std::copy(merged, merged + CUS, cu);
    }
    return cu[CUS - 1];
}

}  // namespace zq3d
