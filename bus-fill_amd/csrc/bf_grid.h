// Launch sizes: which grids HIP takes, and the grids of kernels that cover any
// size.  Plain C++ without HIP: the kernel files include it, and so does the
// CPU check of the plans (tests/plan_check.cpp).
#pragma once

#include <cstdint>

namespace bf {

// HIP launches fewer than 2^32 work items along a dimension.
inline bool launch_fits(int64_t workgroups, int threads) { return workgroups * threads < (int64_t(1) << 32); }

// Workgroups of the wide dequant kernel (one thread per eight weights), 0 where
// that is more than a launch takes (2^35 weights): the general kernel's threads
// step through any size.
inline constexpr int kDequantThreads = 256;
inline int64_t dequant_wide_grid(int N, int K) {
    const int64_t units = (int64_t)N * (K >> 5) * 4, grid = (units + kDequantThreads - 1) / kDequantThreads;
    return launch_fits(grid, kDequantThreads) ? grid : 0;
}

}  // namespace bf
