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

// The one-launch fit of k meshes, the largest of n unknowns, u in all, while
// beside unknowns are fitted next to it: a workgroup takes 0.08 + 0.105 per 1,000
// unknowns, 256 meshes at a time, longer by a share that grows with what the
// meshes in work hold together (their vectors leave the L2 caches).  Measured and estimated, in ms: 256 meshes of 160 unknowns 0.12
// and 0.11, 1,000 of 854 0.86 and 0.79, 600 of 3,694 1.85 and 1.83, 64 of 14,176
// 2.09 and 2.09, 512 of them 5.75 and 5.23, 8 of 56,062 7.2 and 7.4, 256 of them 14.5
// and 13.9.
inline double one_launch_ms(int k, int64_t n, double u, double beside) {
    if (k == 0) return 0.0;
    const int rounds = (k + 255) / 256;
    return rounds * (0.08 + 1.05e-4 * (double)n) * (1.0 + 0.35 * std::sqrt(1e-6 * (u / rounds + beside)));
}
// The many-mesh solver: its chain of launches, by the deepest octree, the meshes
// and the unknowns.  64 meshes of depth 3 and 160 unknowns 0.58 and 0.58, 1,000 of
// 4 and 854 1.82 and 2.08, 512 of 5 and 3,694 2.66 and 3.38, 16 of 6 and 14,176 1.54
// and 1.63, 2 of 7 and 56,062 1.91 and 1.88, 128 of these 10.4 and 10.0.
inline double many_mesh_ms(int meshes, int depth, double u) {
    return meshes ? 0.28 + 0.03 * depth * depth + 3.4e-4 * meshes + 1.15e-6 * u : 0.0;
}

// How many of the meshes that may share the one-launch fit do, the smallest
// first (cand: ascending sizes; big: the meshes that may not).  The others go to
// the many-mesh solver, while that makes the two together faster by these
// estimates, and no more than it takes (most, in all).  The two run side by side,
// but on the CUs that the one launch leaves: with 256 workgroups or more they run
// one after the other (600 meshes of 854 unknowns: all in one launch 0.65 ms, 512
// of them and the others beside it 1.28, which an estimate by the slower one alone
// had chosen; 128 of 56,062: all in the many-mesh solver 10.6, 25 of them in the
// launch beside it 12.2).  24 meshes of 14,282 to 131,176 unknowns: all under the cap in one
// launch 6.1 ms, chosen so 5.0; 2 meshes of 56,062: 6.4 and 1.9.
inline int one_launch_count(const std::vector<SplitMesh>& cand, const std::vector<SplitMesh>& big, int most) {
    double u_many = 0, u_one = 0;
    int depth = 0;
    for (const SplitMesh& m : big) {
        u_many += (double)m.unknowns;
        depth = std::max(depth, m.depth);
    }
    for (const SplitMesh& m : cand) u_one += (double)m.unknowns;
    const int n = (int)cand.size(), nbig = (int)big.size(), least = n - std::min(n, std::max(0, most - nbig));
    int best = n;
    double best_ms = INFINITY;
    for (int k = n; k >= least; --k) {   // the k smallest in one launch
        if (k < n) {
            u_one -= (double)cand[k].unknowns;
            u_many += (double)cand[k].unknowns;
            depth = std::max(depth, cand[k].depth);
        }
        const double one = one_launch_ms(k, k ? cand[k - 1].unknowns : 0, std::max(u_one, 0.0), u_many);
        const double many = many_mesh_ms(nbig + n - k, depth, u_many);
        const double ms = std::max(one, many) + std::min(one, many) * std::min(1.0, k / 256.0);
        if (ms < best_ms) {
            best_ms = ms;
            best = k;
        }
    }
    return best;
}

}  // namespace its
