// Block-wise MFMA GEMM for Q4_0 weights off the fast kernels' grid: K a
// multiple of 32 but not of 256, or operands off their 16-byte boundaries
// (k_gemm_block).
//
//   C[m][n] = sum_b d[n][b] * (sum_{k in b} A[m][k] * (q[n][k] - 8))
//
// One v_mfma_f32_16x16x32_f16 is one 32-weight block of a 16 x 16 output tile:
// the codes enter as the exact integers q - 8, and the block's fp32 sum meets
// its scale in an fp32 FMA, so no weight is rounded (as in k_gemm_simple, which
// served these shapes with one thread per output and two byte loads per
// weight: 1,244 us at M = 37, 3001 x 2336).
//
// A workgroup computes 16 NT weight rows x 16 MT batch rows; its eight waves
// split K and add their sums in wave order through LDS (deterministic).
// Operands come straight from global memory (unaligned 8- and 16-byte loads),
// four blocks in flight per wave.
//
// Measured (Q4_0, us per GEMM, k_gemm_simple -> here): M = 37, 3001 x 2336
// 1244 -> 9.7; M = 1 / 300, 5000 x 5152 1442 / 35,700 -> 20 / 120 (planes
// 1761 -> 12 at M = 1); error against 64-bit sums 8e-7 .. 1.2e-6 -> 0.7e-7 ..
// 1.0e-7.  Bound by the cache lines its row-strided loads touch, not by their
// latency: eight blocks in flight or 4 / 16 waves change nothing, and 4-byte
// code loads with two 8-byte activation loads gain 10 % at M = 1 and lose
// 15-25 % from M = 37.
#include <algorithm>
#include <type_traits>

#include "bf_formats.h"
#include "bf_launch.h"

namespace bf {
namespace {

constexpr int kBkWaves = 8;
constexpr int kBkUnroll = 4;             // blocks in flight per wave

struct __attribute__((packed, aligned(2))) B8a2 { uint32_t x, y; };
struct __attribute__((packed, aligned(2))) B16a2 { uint32_t x, y, z, w; };
struct __attribute__((packed, aligned(1))) B4a1 { uint32_t x; };

// One lane's eight codes of a block (k = 8 g .. 8 g + 7) and the block's scale.
struct BkRaw { uint32_t x, y; uint16_t d; };

template <int QT>
__device__ __forceinline__ BkRaw bk_load(const uint8_t* row, const uint8_t* aux, int b, int g) {
    if constexpr (QT == QT_Q4_0) {                     // bytes 8 (g % 2) .. of the low (g < 2) or high nibbles
        const uint8_t* p = row + 18 * (int64_t)b;
        const B8a2 v = *(const B8a2*)(p + 2 + 8 * (g & 1));
        return BkRaw{v.x, v.y, *(const uint16_t*)p};
    } else {
        return BkRaw{((const B4a1*)(row + 16 * (int64_t)b + 4 * g))->x, 0, *(const uint16_t*)(aux + 2 * (int64_t)b)};
    }
}

// q - 8 of a lane's eight codes, exact in fp16.
template <int QT>
__device__ __forceinline__ h8 bk_codes(const Magic& mg, const BkRaw& r, int g) {
    uint32_t p[4];
    h2 unbias;
    uint32_t mask, bits;
    if constexpr (QT == QT_Q4_0) {
        const int sh = 2 * (g & 2);
        const uint32_t x = r.x >> sh, y = r.y >> sh;
        p[0] = perm_b32(x, x, SEL_B01);
        p[1] = perm_b32(x, x, SEL_B23);
        p[2] = perm_b32(y, y, SEL_B01);
        p[3] = perm_b32(y, y, SEL_B23);
        unbias = h2{(_Float16)-1032.0f, (_Float16)-1032.0f};
        mask = mg.lo_mask;
        bits = mg.lo_bits;
    } else {
        p[0] = perm_b32(r.x, r.x, SEL_BB0);
        p[1] = perm_b32(r.x, r.x, SEL_BB1);
        p[2] = perm_b32(r.x, r.x, SEL_BB2);
        p[3] = perm_b32(r.x, r.x, SEL_BB3);
        unbias = h2{(_Float16)-1032.0f, (_Float16)-72.0f};
        mask = mg.pl_mask;
        bits = mg.pl_bits;
    }
    h8 o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const h2 v = as_h2(and_or(p[i], mask, bits)) + unbias;
        o[2 * i] = v[0];
        o[2 * i + 1] = v[1];
    }
    return o;
}

template <int QT, int MT, int NT>
__global__ __launch_bounds__(64 * kBkWaves)
void k_gemm_block(const uint8_t* __restrict__ W, const uint8_t* __restrict__ Waux, const uint16_t* __restrict__ A,
                  int lda, void* __restrict__ C, int ldc, int out_f16, int M, int N, int K, int nb) {
    __shared__ f4 sums[kBkWaves][MT * NT][64];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int mc = (int)blockIdx.x / nb, m0 = 16 * MT * mc;
    const int64_t n0 = 16 * NT * (int64_t)((int)blockIdx.x - mc * nb);
    const int blocks = K >> 5, b0 = wave * blocks / kBkWaves, b1 = (wave + 1) * blocks / kBkWaves;
    const uint8_t* row[NT];
    const uint8_t* aux[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int64_t n = min(n0 + 16 * t + r, (int64_t)N - 1);
        row[t] = W + n * (QT == QT_Q4_0 ? 18 * (int64_t)blocks : 16 * (int64_t)blocks);
        aux[t] = QT == QT_Q4_0 ? nullptr : Waux + 2 * n * blocks;
    }
    const uint16_t* act[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) act[t] = A + (int64_t)min(m0 + 16 * t + r, M - 1) * lda + 8 * g;
    const Magic mg = make_magic();
    f4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[i][t] = f4{0.f, 0.f, 0.f, 0.f};

    auto pass = [&](auto count, int b) {
        constexpr int U = decltype(count)::value;
        BkRaw w[U][NT];
        B16a2 a[U][MT];
#pragma unroll
        for (int u = 0; u < U; u++) {
#pragma unroll
            for (int t = 0; t < NT; t++) w[u][t] = bk_load<QT>(row[t], aux[t], b + u, g);
#pragma unroll
            for (int i = 0; i < MT; i++) a[u][i] = *(const B16a2*)(act[i] + 32 * (int64_t)(b + u));
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const h8 q = bk_codes<QT>(mg, w[u][t], g);
                const float d = half_bits_to_float(w[u][t].d);
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const h8 x = __builtin_bit_cast(h8, u4{a[u][i].x, a[u][i].y, a[u][i].z, a[u][i].w});
                    const f4 p = mfma16x16x32(x, q, f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[i][t][e] = __builtin_fmaf(d, p[e], acc[i][t][e]);
                }
            }
    };
    int b = b0;
    for (; b + kBkUnroll <= b1; b += kBkUnroll) pass(std::integral_constant<int, kBkUnroll>(), b);
    for (; b < b1; b++) pass(std::integral_constant<int, 1>(), b);

#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++) sums[wave][i * NT + t][lane] = acc[i][t];
    __syncthreads();
    // thread -> (tile, lane's four outputs): rows 4 g .. 4 g + 3, column r
    for (int x = (int)threadIdx.x; x < MT * NT * 64; x += 64 * kBkWaves) {
        const int tile = x >> 6, i = tile / NT, t = tile - i * NT;
        f4 s = sums[0][tile][lane];
#pragma unroll
        for (int w = 1; w < kBkWaves; w++) s += sums[w][tile][lane];
        const int64_t n = n0 + 16 * t + r;
        if (n >= N) continue;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int m = m0 + 16 * i + 4 * g + e;
            if (m >= M) break;
            const int64_t o = (int64_t)m * ldc + n;
            if (out_f16) ((_Float16*)C)[o] = (_Float16)s[e];
            else ((float*)C)[o] = s[e];
        }
    }
}

struct BlockPlan { int MT, NT, nb; int64_t grid; };

// Batch rows of a workgroup: all of them up to 64.  Two 16-row weight tiles
// per workgroup (each activation load feeds two MFMAs) from 300 single ones on:
// 313 (5000 rows, M = 1 / 8 / 20) 21.4 / 23.9 / 28.7 -> 20.4 / 21.5 / 24.6 us,
// 1,565 (M = 300) 145 -> 120; 250 (2000 rows, M = 128) 18.6 -> 25.9.
BlockPlan plan_block(const GemmArgs& g) {
    BlockPlan p;
    p.MT = std::min(4, (g.M + 15) / 16);
    const int64_t mcs = (g.M + 16 * p.MT - 1) / (16 * p.MT), n16 = ((int64_t)g.N + 15) / 16;
    p.NT = mcs * n16 >= 300 ? 2 : 1;
    p.nb = (int)((n16 + p.NT - 1) / p.NT);
    p.grid = mcs * p.nb;
    return p;
}

template <int QT, int MT>
hipError_t launch_block(const GemmArgs& g, const BlockPlan& p, hipStream_t st) {
    auto k = p.NT == 2 ? k_gemm_block<QT, MT, 2> : k_gemm_block<QT, MT, 1>;
    hipLaunchKernelGGL(k, dim3((unsigned)p.grid), dim3(64 * kBkWaves), 0, st, g.W, g.Waux, g.A, g.lda, g.C, g.ldc,
                       g.out_f16, g.M, g.N, g.K, p.nb);
    return hipGetLastError();
}

template <int QT>
hipError_t dispatch_block(const GemmArgs& g, const BlockPlan& p, hipStream_t st) {
    if (p.MT == 1) return launch_block<QT, 1>(g, p, st);
    if (p.MT == 2) return launch_block<QT, 2>(g, p, st);
    if (p.MT == 3) return launch_block<QT, 3>(g, p, st);
    return launch_block<QT, 4>(g, p, st);
}

}  // namespace

bool block_supports(const GemmArgs& g) {
    return (g.qtype == QT_Q4_0 || g.qtype == QT_PLANES) && g.K % 32 == 0 && plan_block(g).grid < (int64_t(1) << 31);
}

hipError_t gemm_block(const GemmArgs& g, hipStream_t st) {
    const BlockPlan p = plan_block(g);
    return g.qtype == QT_Q4_0 ? dispatch_block<QT_Q4_0>(g, p, st) : dispatch_block<QT_PLANES>(g, p, st);
}

}  // namespace bf
