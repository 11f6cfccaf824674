// Launch arithmetic of its_amd/csrc/launch.hpp: blocks of strided launches.
#include <cstdio>
#include <cstdlib>

#include "launch.hpp"

int main(int argc, char** argv) {   // items per_block threads, repeated
    for (int k = 1; k + 2 < argc; k += 3)
        std::printf("%u\n", its::strided_blocks(std::atoll(argv[k]), std::atoll(argv[k + 1]), std::atoi(argv[k + 2])));
    return 0;
}
