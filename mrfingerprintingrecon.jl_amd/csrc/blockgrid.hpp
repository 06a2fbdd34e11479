// Grid dimensions of launches of very many blocks, kept free of HIP so that
// they can be tested on the host.
#pragma once

#include <cstdint>

namespace msr {

struct BlockGrid {
    unsigned x, y;
};

// n >= 1 blocks of `threads` threads as a grid (x, y) with x y >= n: one row
// while it fits.  A launch takes less than 2^32 threads per dimension, which
// one block of 256 per 4 x 4 x 4 cells reaches at a grid of 1024 x 1024 x 1024.
// Block (bx, by) is number by * x + bx; those from n on have no work.
inline BlockGrid split_blocks(int64_t n, int threads) {
    const int64_t most = ((int64_t)1 << 31) / threads;
    const int64_t y = (n + most - 1) / most;
    return {(unsigned)((n + y - 1) / y), (unsigned)y};
}

}  // namespace msr
