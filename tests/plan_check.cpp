// CPU check of the kernels' plans and grids (bus-fill_amd/csrc/bf_grid.h,
// bf_block_plan.h, bf_tile_plan.h).
// Every check prints what it expected on failure; exit status 0 when all hold.
// `plan_check tile M N K` and `plan_check block M N K` print a plan on 256 CUs
// (TA NB F R S, with the scratch of a 128-row dense launch, and whether a format
// of factor 1 would take 128-row launches instead; MT NT NW).
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "bf_block_plan.h"
#include "bf_grid.h"
#include "bf_tile_plan.h"

using namespace bf;

namespace {

int failures = 0;

void expect(bool ok, const char* what, int64_t a = 0, int64_t b = 0, int64_t c = 0) {
    if (ok) return;
    failures++;
    std::printf("FAIL %s (%lld, %lld, %lld)\n", what, (long long)a, (long long)b, (long long)c);
}

constexpr int64_t kItems = int64_t(1) << 32;           // work items of a launch along a dimension: fewer

// The wide dequant grid covers every weight, is one HIP takes, and is given up
// (for the general kernel) only where no such grid exists.
void check_dequant() {
    const int shapes[][2] = {{1, 32},        {17408, 5120},    {1 << 19, 1 << 15},  {1 << 20, 1 << 15},
                             {1 << 25, 992}, {1 << 25, 1024},  {(1 << 25) - 1, 1024}, {(1 << 25) + 1, 1024},
                             {1 << 30, 256}, {1 << 30, 8192},  {2147483647, 32}};
    for (const auto& s : shapes) {
        const int64_t weights = (int64_t)s[0] * s[1], need = (weights / 8 + 255) / 256, grid = dequant_wide_grid(s[0], s[1]);
        if (need * 256 < kItems) expect(grid == need, "dequant grid covers the weights", s[0], s[1], grid);
        else expect(grid == 0, "dequant grid above the launch limit", s[0], s[1], grid);
    }
}

// The block-wise kernel's workgroups cover the outputs, and a grid that HIP does
// not take (64 kBkWaves threads per workgroup) is given up.
void check_block_grid() {
    const int shapes[][3] = {{1, 1, 32},          {37, 3001, 2336},     {300, 5000, 5152},   {129, 2800, 1184},
                             {1, 1 << 28, 32},    {1, 1 << 27, 32},     {1, (1 << 28) - 32, 32}, {2147483647, 16, 32},
                             {200000, 200000, 32}, {1 << 20, 1 << 13, 32}, {1 << 20, 1 << 16, 64}};
    for (const auto& s : shapes) {
        const int M = s[0], N = s[1];
        const BlockPlan p = plan_block(M, N, s[2], 256);
        const int64_t rows = 16 * (int64_t)(p.NT ? p.NT : p.NW), cols = ((int64_t)N + rows - 1) / rows;
        expect(p.MT >= 1 && p.MT <= 4 && p.grid % cols == 0 && p.grid / cols * 16 * p.MT >= M, "block grid covers", M, N, p.grid);
        const bool fits = launch_fits(p.grid, 64 * kBkWaves);
        expect(fits == (p.grid * 64 * kBkWaves < kItems), "block grid against the launch limit", M, N, p.grid);
    }
    expect(!launch_fits(plan_block(1, 1 << 28, 32, 256).grid, 64 * kBkWaves), "2^28 weight rows: more than a launch");
    expect(launch_fits(plan_block(1, (1 << 28) - 32, 32, 256).grid, 64 * kBkWaves), "2^28 - 32 weight rows: a launch");
}

// Every tile plan covers the outputs, keeps its partials within the scratch on
// offer and makes a grid that HIP takes; above that there is no plan.
void check_tile_grid() {
    const size_t offers[] = {0, size_t(1) << 20, size_t(32) << 20};
    const int Ms[] = {129, 192, 257, 2000, 100000, 1 << 22, 1 << 24, 1 << 28, 2147483647}, Ns[] = {1, 128, 5120, 17408, 1 << 20, 1 << 28},
              Ks[] = {256, 1280, 17408};
    for (const size_t scratch : offers)
        for (const int M : Ms)
            for (const int N : Ns)
                for (const int K : Ks) {
                    TilePlan p{};
                    if (!plan_tile(M, N, K, 256, scratch, p)) {
                        const int64_t least = ((int64_t)M + 255) / 256 * (((int64_t)N + 255) / 256);
                        expect((least + 16 * 256) * kTlThreads >= kItems, "no tile plan", M, N, K);
                        continue;
                    }
                    const int64_t T = (int64_t)p.mt * (((int64_t)N + 128 * p.NB - 1) / (128 * p.NB));
                    expect(p.F + (int64_t)p.R == T && (int64_t)p.mt * 64 * p.TA >= M, "tiles cover", M, N, K);
                    expect(p.S >= 1 && p.S <= std::min(16, K / 256) && p.part <= scratch && (p.S == 1) == (p.part == 0),
                           "tile cuts", M, N, K);
                    expect((p.F + (int64_t)p.R * p.S) * kTlThreads < kItems, "tile grid against the launch limit", M, N, K);
                }
}

// The block-wise kernel only where it is the faster one.
void check_block_choice() {
    expect(block_slower(1, 262144, 32) && block_slower(1, 1000000, 32), "one row, one block, many weight rows: a thread per output");
    for (const int M : {1, 2, 16, 300})
        for (const int N : {16, 5000, 131072})
            for (const int K : {32, 64, 2336}) expect(!block_slower(M, N, K), "block-wise", M, N, K);
    expect(!block_slower(2, 1000000, 32) && !block_slower(1, 1000000, 64), "two rows or two blocks: block-wise");
}

// Tiles or 128-row launches, at measured points on both sides of the rule (256
// CUs, 32 MB of scratch; formats by their factor).
void check_tile_choice() {
    const double q4k = 1.04, q40 = 1.08, planes = 1.12;
    struct Point { int M, N, K; double slow; bool slices; };
    const Point points[] = {
        {129, 17408, 5120, q4k, true},    {136, 17408, 5120, q4k, true},    {192, 17408, 5120, q4k, false},
        {160, 17408, 5120, q40, true},    {192, 17408, 5120, q40, false},   {193, 17408, 5120, planes, true},
        {256, 17408, 5120, q4k, false},   {257, 17408, 5120, planes, false}, {160, 17408, 17408, q4k, true},
        {193, 17408, 17408, q4k, true},   {256, 17408, 17408, q40, false},  {129, 28672, 4096, planes, false},
        {129, 32000, 4096, q4k, false},   {144, 16384, 4096, q40, false},   {160, 16896, 2816, planes, false},
        {129, 5120, 5120, q4k, true},     {140, 5120, 5120, q4k, false},    {132, 2048, 8192, planes, true},
        {136, 2048, 8192, q4k, false},    {136, 6144, 4096, q40, true},     {144, 4096, 4096, q4k, false},
        {129, 1024, 1024, q4k, false},    {129, 256, 17408, planes, false}, {129, 5120, 17408, q4k, false},
        {129, 4042, 3328, q40, false},    {512, 17408, 5120, planes, false}, {256, 2048, 8192, q4k, false},
        {300, 5120, 5120, q4k, false},    {129, 8870, 4864, q4k, false},    {130, 11921, 1792, planes, false},
        {2000, 17408, 17408, q4k, false}};
    for (const Point& x : points) {
        TilePlan p{};
        expect(plan_tile(x.M, x.N, x.K, 256, size_t(32) << 20, p), "a tile plan", x.M, x.N, x.K);
        expect(slices_faster(x.M, x.N, x.K, 256, x.slow, p) == x.slices, x.slices ? "128-row launches" : "tiles", x.M, x.N, x.K);
    }
}

}  // namespace

int main(int argc, char** argv) {
    if (argc == 5) {
        const int M = std::atoi(argv[2]), N = std::atoi(argv[3]), K = std::atoi(argv[4]);
        if (!std::strcmp(argv[1], "block")) {
            const BlockPlan b = plan_block(M, N, K, 256);
            std::printf("%d %d %d\n", b.MT, b.NT, b.NW);
            return 0;
        }
        TilePlan p{};
        const int64_t units = ((int64_t)N + 127) / 128 * (K / 256);
        if (!plan_tile(M, N, K, 256, (size_t)std::min<int64_t>(units, 256) * 2 * 128 * 128 * 4, p)) return 1;
        std::printf("%d %d %d %d %d %d\n", p.TA, p.NB, p.F, p.R, p.S, (int)slices_faster(M, N, K, 256, 1.0, p));
        return 0;
    }
    const char* only = argc > 1 ? argv[1] : "";
    auto on = [&](const char* name) { return !*only || !std::strcmp(only, name); };
    if (on("dequant")) check_dequant();
    if (on("block_grid")) check_block_grid();
    if (on("block_choice")) check_block_choice();
    if (on("tile_grid")) check_tile_grid();
    if (on("tile_choice")) check_tile_choice();
    if (!failures) std::printf("ok\n");
    return failures != 0;
}
