// Which meshes of a batch share the one-launch fit, plain C++ (no HIP headers).
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

namespace its {

struct SplitMesh {
    int64_t unknowns;
    int depth;
};

// How many of the meshes that may share the one-launch fit do, the smallest
// first (cand: ascending sizes; big: the meshes that may not).  The others go to
// the many-mesh solver, while that makes the slower of the two, which run side by
// side, faster, and no more than it takes (most, in all).  Estimates, in ms,
// from measured fits:
//   - one workgroup takes 0.17 + 0.2 per 1,000 unknowns, 256 meshes at a
//     time (0.19 ms at 160 unknowns, 0.66 at 3,668, 1.97 at 14,110, 6.1 at
//     31,101 with more iterations, 8.7 at 55,852);
//   - the many-mesh solver takes 0.055 depth^2 for its chain of launches
//     (0.83 ms at depth 3, 1.8 at 6, 2.7 at 7) and 1.1 per million unknowns
//     in all (5.8 ms for 256 meshes of 14,110).
// 24 meshes of 14,282 to 131,176 unknowns: all under the cap in one launch
// 6.1 ms, chosen so 5.0; 6 meshes of 7,165 to 55,852: 8.7 and 2.7.
inline int one_launch_count(const std::vector<SplitMesh>& cand, const std::vector<SplitMesh>& big, int most) {
    double unknowns = 0;
    int depth = 0;
    for (const SplitMesh& m : big) {
        unknowns += (double)m.unknowns;
        depth = std::max(depth, m.depth);
    }
    const int n = (int)cand.size(), least = n - std::min(n, std::max(0, most - (int)big.size()));
    int best = n;
    double best_ms = INFINITY;
    for (int k = n; k >= least; --k) {   // the k smallest in one launch
        if (k < n) {
            unknowns += (double)cand[k].unknowns;
            depth = std::max(depth, cand[k].depth);
        }
        const double one = k ? (0.17 + 2e-4 * (double)cand[k - 1].unknowns) * ((k + 255) / 256) : 0.0;
        const double many = unknowns > 0 ? 0.055 * depth * depth + 1.1e-6 * unknowns : 0.0;
        const double ms = std::max(one, many);
        if (ms < best_ms) {
            best_ms = ms;
            best = k;
        }
    }
    return best;
}

}  // namespace its
