// Launch grids.
#pragma once

#include <cstdint>

namespace mb {

// Blocks (x) of a launch that wants `want` of them: a dimension holds fewer
// than 2^32 threads (the runtime launches the remainder modulo 2^32, without
// an error), so kernels whose blocks grow with the data stride over what one
// launch leaves.
constexpr unsigned launch_blocks(int64_t want, int threads) {
    const int64_t most = (((int64_t)1 << 32) - 1) / threads;
    return (unsigned)(want < 1 ? 1 : want < most ? want : most);
}

}  // namespace mb
