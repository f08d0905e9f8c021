// Plan of the tile kernel (bf_gemm_tile.hip).  Plain C++ without HIP: the
// kernel file includes it, and so does the CPU check of the plans
// (tests/plan_check.cpp).
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "bf_grid.h"

namespace bf {

inline constexpr int kTlThreads = 512;   // eight waves, two per SIMD

struct TilePlan {
    int TA, NB, mt, F, R, S;
    size_t part;                         // workspace bytes
    double cost;                         // tile_cost, us
};

// Microseconds of a plan, from measured launches (Q4_K): a super-group of each
// tile shape takes `lo` up to 0.4 of the CUs busy and up to `hi` with all of
// them (with fewer busy CUs the chip clocks higher), a round 6.5
// for its start and end; the cut tiles' partials are written and read once,
// and their sum is a launch of its own.
inline double tile_cost(int TA, int NB, int nsg, int cus, int F, int R, int S, size_t piece) {
    const double lo = NB == 2 ? 4.9 : TA == 4 ? 2.95 : TA == 3 ? 2.45 : 2.2;
    const double hi = NB == 2 ? 7.6 : TA == 4 ? 4.1 : TA == 3 ? 3.3 : 2.4;
    const int units = R * S, full = units / cus, rem = units % cus, n = (nsg + S - 1) / S;
    const double last = lo + (hi - lo) * std::max(0.0, ((double)rem / cus - 0.4) / 0.6);
    double c = F / cus * (nsg * hi + 6.5) + full * (n * hi + 6.5) + (rem ? n * last + 6.5 : 0.0);
    if (S > 1) c += 3.0 + 2.0 * (double)units * (double)piece / 8e6;
    return c;
}

// The plan of least cost whose partials fit `scratch` bytes; false where the
// tile kernel does not serve the shape.
inline bool plan_tile(int M, int N, int K, int cus, size_t scratch, TilePlan& p) {
    if (M <= 128 || K % 256 || N < 1) return false;
    const int nsg = K / 256;
    double best = 0;
    for (int NB = 2; NB >= 1; NB--)
        for (int TA = 4; TA >= (NB == 2 ? 4 : 2); TA--) {
            const int64_t mt = ((int64_t)M + 64 * TA - 1) / (64 * TA), T = mt * (((int64_t)N + 128 * NB - 1) / (128 * NB));
            if (!launch_fits(T + 16 * cus, kTlThreads)) continue;      // (fewer than 16 cus more units than tiles)
            const int F = (int)(T / cus * cus), R = (int)T - F;
            const size_t piece = (size_t)64 * TA * 128 * NB * 4;
            for (int S = 1; S <= std::min(nsg, 16); S++) {
                if (S > 1 && (R == 0 || (size_t)R * S * piece > scratch)) break;
                const double cost = tile_cost(TA, NB, nsg, cus, F, R, S, piece);
                if (best == 0 || cost < best) {
                    best = cost;
                    p = TilePlan{TA, NB, (int)mt, F, R, S, S > 1 ? (size_t)R * S * piece : 0, cost};
                }
            }
        }
    return best > 0;
}

// Microseconds of the same call as dense launches of 128 rows (shares of the
// 128 x 256 weight units, one workgroup per CU) and one of the remaining rows,
// on whichever kernel serves those; measured, all formats.
inline double slices_cost(int M, int N, int K, int cus) {
    const double units = (double)((((int64_t)N + 127) / 128 * (K / 256) + cus - 1) / cus), w = (double)N * K / 1e6;
    const int r = M % 128;
    const double rest = r == 0 ? 0.0 : r <= 8 ? 3.6 + 0.15 * w : r <= 32 ? 5.0 + 0.155 * w : r <= 64 ? 9.3 + 0.19 * w
                        : r <= 96 ? 9.5 + 0.26 * w : 10.7 + 0.32 * w;
    return M / 128 * (9.0 + 2.75 * units) + rest;
}

// Up to 256 rows, where 128-row launches beat the plan.  `slow`: the format's
// super-groups against tile_cost's, which are Q4_K's on a chip that is not half
// idle (Q4_K 1.04, Q4_0 1.08, planes 1.12).
// * Uncut tiles (64 TA x 128, TA >= 3) on little more than half the CUs, and
//   whole rounds with a cut remainder behind them at K >= 8192: where the costs
//   say so.  17408 x 5120 at M = 132 / 160 / 224 / 256, slices and tiles, us:
//   planes 51.8 / 57.7 / 69.4 / 75.0 and 61.3 / 62.1 / 76.8 / 78.1, Q4_K 52.0 /
//   59.4 / 71.2 / 77.7 and 56.2 / 55.8 / 68.5 / 70.8; 17408 x 17408 at M = 160:
//   planes 145 and 184, Q4_K 152 and 173.
// * One dense launch and at most 8 rows (4 on longer K) of a matrix that its
//   workgroups share evenly, against tiles cut in four or more: 6144 x 4096
//   planes / Q4_K at M = 130 24.4 / 24.7 and 26.3 / 25.6, 2048 x 8192 at M = 129
//   21.1 / 21.1 and 23.1 / 22.6.
// Over 7143 measured shapes, batches and formats the tiles alone were slower by
// more than 2 % at 758, up to 1.37 times; with this rule at 24, up to 1.07 times
// (weights of 2^28 and more), for 134 where they would have been 2-16 % faster.
inline bool slices_faster(int M, int N, int K, int cus, double slow, const TilePlan& p) {
    if (M > 256) return false;
    const int64_t units = ((int64_t)N + 127) / 128 * (K / 256);
    if (M % 128 <= (K <= 6144 ? 8 : 4) && M < 256 && N % 128 == 0 && N >= 2048 && p.F == 0 && p.S >= 4 &&
        4 * units >= 7 * cus && 4 * units <= 13 * cus)
        return true;
    if (K < 3072) return false;
    const bool half_idle = p.F == 0 && p.S == 1 && 2 * p.R > cus && p.TA >= 3, spills = p.F > 0 && K >= 8192;
    return (half_idle || spills) && slices_cost(M, N, K, cus) < (spills ? 1.04 : slow) * p.cost;
}

}  // namespace bf
