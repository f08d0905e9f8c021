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
};

// Microseconds of a plan, from measured launches (Q4_K): a super-group of each
// tile shape takes `lo` up to 0.4 of the CUs busy and up to `hi` with all of
// them (the chip is bound by power: fewer busy CUs clock higher), a round 6.5
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
                    p = TilePlan{TA, NB, (int)mt, F, R, S, S > 1 ? (size_t)R * S * piece : 0};
                }
            }
        }
    return best > 0;
}

}  // namespace bf
