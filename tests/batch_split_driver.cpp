// its_amd/csrc/batch_split.hpp on the command line: most, number of meshes
// above the cap, then unknowns and depth of every mesh (those first).
#include <cstdio>
#include <cstdlib>

#include "batch_split.hpp"

int main(int argc, char** argv) {
    const int most = std::atoi(argv[1]), nbig = std::atoi(argv[2]);
    std::vector<its::SplitMesh> big, cand;
    for (int k = 3; k + 1 < argc; k += 2)
        ((int)big.size() < nbig ? big : cand).push_back({std::atoll(argv[k]), std::atoi(argv[k + 1])});
    std::printf("%d\n", its::one_launch_count(cand, big, most));
    return 0;
}
