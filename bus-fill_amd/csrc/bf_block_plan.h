// Plan of the block-wise GEMM (bf_gemm_block.hip).  Plain C++ without HIP: the
// kernel file includes it, and so does the CPU check of the plans
// (tests/plan_check.cpp).
#pragma once

#include <algorithm>
#include <cstdint>

#include "bf_grid.h"

namespace bf {

inline constexpr int kBkWaves = 8;       // waves of a workgroup

// 16-row batch tiles and weight tiles of a workgroup, the staged form's waves
// over weight rows, workgroups.  NT = 0: the staged form, nb its batch chunks.
struct BlockPlan { int MT, NT, NW, nb; int64_t grid; };

// Batch rows of a workgroup: all of them up to 64.  Two 16-row weight tiles
// per workgroup (each activation load feeds two MFMAs) from 300 single ones on:
// 313 (5000 rows, M = 1 / 8 / 20) 21.4 / 23.9 / 28.7 -> 20.4 / 21.5 / 24.6 us;
// 250 (2000 rows, M = 128) 18.6 -> 25.9.
//
// The staged form from 33 rows, where those tiles (64 batch rows x 32 weight
// rows) take more than a workgroup per CU: 5000 x 5152 Q4_0 at M = 64 / 80 (157
// / 314 tiles) 32.3 / 51 us direct, 35 / 32 staged; 4000 x 2976 at M = 128 / 129
// (250 / 375) 19.7 / 32 and 22.5 / 20.  Short K from 1.5 per CU: 4500 x 672 at
// M = 100 / 129 (282 / 423) 9.7 / 10.1 and 10.7 / 9.9.  Two groups of four waves
// where their grid fits a round: 5000 x 5152 at M = 129 (237) 32 us, eight
// waves 47; at M = 200 (316) 67 and 51.
inline BlockPlan plan_block(int M, int N, int K, int cus) {
    BlockPlan p;
    const int64_t m16 = ((int64_t)M + 15) / 16, n16 = ((int64_t)N + 15) / 16;
    p.MT = (int)std::min<int64_t>(4, m16);
    const int64_t mcs = (m16 + p.MT - 1) / p.MT, direct = mcs * ((n16 + 1) / 2);
    if (M > 32 && direct > cus && (K >= 1024 || 2 * direct > 3 * cus)) {
        p.MT = (int)((m16 + mcs - 1) / mcs);           // equal chunks
        p.NT = 0;
        p.NW = mcs * (((int64_t)N + 63) / 64) <= cus ? 4 : 8;
        p.nb = (int)mcs;
        p.grid = mcs * (((int64_t)N + 16 * p.NW - 1) / (16 * p.NW));
        return p;
    }
    p.NW = kBkWaves;
    p.NT = mcs * n16 >= 300 ? 2 : 1;
    p.nb = (int)((n16 + p.NT - 1) / p.NT);
    p.grid = mcs * p.nb;
    return p;
}

// One block per weight row and one batch row: from some 2^18 weight rows on, a
// thread per output is faster (Q4_0 / planes, a thread per output against here,
// us: 131072 rows 7.5 / 9.4 and 7.2 / 7.0, 262144 rows 11.8 / 12.9 and 14.6 /
// 14.4, 1000000 rows 39 / 40 and 52 / 49; at two batch rows 73 / 76 and 56 / 53).
inline bool block_slower(int M, int N, int K) { return M == 1 && K == 32 && N >= 200000; }

}  // namespace bf
