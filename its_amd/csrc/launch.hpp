// Launch arithmetic of the ITS gfx950 library, plain C++ (no HIP headers).
#pragma once
#include <algorithm>
#include <cstdint>

namespace its {

// A launch dimension holds fewer than 2^32 work items.  Blocks of a launch
// whose kernel strides over the grid: one per `per_block` items, as many as
// that limit leaves.
inline unsigned strided_blocks(int64_t items, int64_t per_block, int threads) {
    const int64_t most = ((int64_t(1) << 32) - 1) / threads;
    return (unsigned)std::min<int64_t>(std::max<int64_t>((items + per_block - 1) / per_block, 1), most);
}

}  // namespace its
