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
//
// Where that takes more than a round of workgroups, k_gemm_block_staged passes
// the activations through LDS (below).
#include <type_traits>

#include "bf_block_plan.h"
#include "bf_formats.h"
#include "bf_launch.h"
#include "bf_lds.h"

namespace bf {
namespace {

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

__device__ __forceinline__ void store_out(float y, void* C, int64_t o, int out_f16) {
    if (out_f16) ((_Float16*)C)[o] = (_Float16)y;
    else ((float*)C)[o] = y;
}

// Outputs of weight row n just stored (batch rows row_of(0) .. row_of(count - 1)):
// the infinite ones with what weights of infinite scale add to them one by one --
// NaN where a code is 8 or the terms have both signs, where the block's sum times
// its scale is an infinity.  (An output that is NaN needs no second look: these
// weights give NaN too.)  After the stores, so the loops stay as they are: there
// the check cost up to 30 % (17408 x 2336 at M = 300, 66 -> 85 us).
template <int QT, class RowOf>
__device__ __forceinline__ void add_infinite_scales(int count, RowOf row_of, const uint8_t* W, const uint8_t* Waux,
                                                    const uint16_t* A, int lda, void* C, int ldc, int out_f16, int M,
                                                    int64_t n, int blocks) {
    const uint8_t* const row = W + n * (QT == QT_Q4_0 ? 18 : 16) * (int64_t)blocks;
#pragma unroll 1
    for (int i = 0; i < count; i++) {
        const int m = row_of(i);
        if (m >= M) continue;
        const uint16_t* const a = A + (int64_t)m * lda;
        const int64_t o = (int64_t)m * ldc + n;
        float y = out_f16 ? (float)((const _Float16*)C)[o] : ((const float*)C)[o];
        if (!__builtin_isinf(y)) continue;
#pragma unroll 1
        for (int k = 0; k < 32 * blocks; k++) {
            const uint8_t* const codes = row + (QT == QT_Q4_0 ? 18 * (int64_t)(k >> 5) + 2 : 16 * (int64_t)(k >> 5));
            const float d = half_bits_to_float(
                *(const uint16_t*)(QT == QT_Q4_0 ? codes - 2 : Waux + 2 * (n * blocks + (k >> 5))));
            if (__builtin_isfinite(d)) {
                k |= 31;
                continue;
            }
            const uint32_t c = codes[QT == QT_Q4_0 ? k & 15 : (k & 31) >> 1];
            const int q = (QT == QT_Q4_0 ? k & 16 : k & 1) ? c >> 4 : c & 15;
            y = __builtin_fmaf((float)__builtin_bit_cast(_Float16, a[k]), (float)(q - 8) * d, y);
        }
        store_out(y, C, o, out_f16);
    }
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
        const int mr = m0 + 16 * i + 4 * g;
        bool inf = false;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (mr + e >= M) break;
            store_out(s[e], C, (int64_t)(mr + e) * ldc + n, out_f16);
            inf |= __builtin_isinf(s[e]);
        }
        if (inf)
            add_infinite_scales<QT>(4, [&](int e) { return mr + e; }, W, Waux, A, lda, C, ldc, out_f16, M, n, blocks);
    }
}

// The staged form: a workgroup computes 16 MT batch rows x 16 NW weight rows (a
// wave 16 of them), K in steps of four blocks.  The activations of a step go
// through LDS, loaded four steps ahead in 16-byte pieces along the rows, so
// each is read once per 64 or 128 weight rows instead of 16 or 32; four lanes
// load a weight row's four blocks whole (two loads where block by block takes
// eight) and swap them by permlane.  NW = 4: two groups of four waves halve K.
//
// Measured (us per GEMM, k_gemm_block -> here, Q4_0 / planes): 5000 x 5152 at
// M = 300 120 / 89 -> 55 / 41, M = 129 62 / 47 -> 32 / 22, M = 80 51 / 36 ->
// 32 / 22; 3001 x 2336 at M = 300 31 / 25 -> 20 / 16; 4500 x 672 at M = 300
// 15.9 / 13.3 -> 13.0 / 10.5.  Error against 64-bit sums 0.9e-7 .. 2.3e-7 (the
// one-thread-per-output kernel 8e-7 .. 1.2e-6).  Bound by a wave's own chain
// of 200-220 instructions per step: eight waves on the same rows take as long
// as four, and halving K over two groups of waves gains where halving the rows
// does not.  Loads under a branch drained all of them at every step (60 us).
constexpr int kStBlocks = 4;             // blocks of a step
constexpr int kStAhead = 4;              // steps whose loads are in flight

struct __attribute__((packed, aligned(1))) B16a1 { uint32_t x, y, z, w; };

// Lane (r, g) of a wave holds block b + g of its weight row: four words of
// codes and the scale (four lanes' loads cover a row's 72 or 64 bytes).
struct StRaw { uint32_t w[4]; uint16_t d; };

template <int QT>
__device__ __forceinline__ StRaw st_load(const uint8_t* row, const uint8_t* aux, int b) {
    StRaw o;
    if constexpr (QT == QT_Q4_0) {
        const uint8_t* p = row + 18 * (int64_t)b;
        const B16a2 v = *(const B16a2*)(p + 2);
        o.w[0] = v.x; o.w[1] = v.y; o.w[2] = v.z; o.w[3] = v.w;
        o.d = *(const uint16_t*)p;
    } else {
        const B16a1 v = *(const B16a1*)(row + 16 * (int64_t)b);
        o.w[0] = v.x; o.w[1] = v.y; o.w[2] = v.z; o.w[3] = v.w;
        o.d = *(const uint16_t*)(aux + 2 * (int64_t)b);
    }
    return o;
}

// Rows of 16 lanes: (a0 a1 a2 a3), (b0 b1 b2 b3) -> (a0 a1 b0 b1), (a2 a3 b2 b3)
__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {
    const auto v = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = v[0];
    b = v[1];
}
// (a0 a1 a2 a3), (b0 b1 b2 b3) -> (a0 b0 a2 b2), (a1 b1 a3 b3)
__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {
    const auto v = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = v[0];
    b = v[1];
}

// Block u of the step for every lane: word g of its codes in x[u] and its scale
// in d[u] (a 4 x 4 transpose over the lane rows, and a broadcast of each).
__device__ __forceinline__ void st_spread(const StRaw& r, uint32_t (&x)[4], float (&d)[4]) {
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = r.w[i];
    swap32(x[0], x[2]);
    swap32(x[1], x[3]);
    swap16(x[0], x[1]);
    swap16(x[2], x[3]);
    uint32_t a = __builtin_bit_cast(uint32_t, half_bits_to_float(r.d)), c = a;
    swap32(a, c);                                      // (d0 d1 d0 d1), (d2 d3 d2 d3)
    uint32_t b = a, e = c;
    swap16(a, b);
    swap16(c, e);
    d[0] = __builtin_bit_cast(float, a);
    d[1] = __builtin_bit_cast(float, b);
    d[2] = __builtin_bit_cast(float, c);
    d[3] = __builtin_bit_cast(float, e);
}

// q - 8 of word g of a block.  Q4_0: k = 4 g .. 4 g + 3 and 16 + 4 g .. (the
// order the activations take in LDS); planes: k = 8 g .. 8 g + 7.
template <int QT>
__device__ __forceinline__ h8 st_codes(const Magic& mg, uint32_t x) {
    if constexpr (QT == QT_PLANES) {
        return bk_codes<QT_PLANES>(mg, BkRaw{x, 0, 0}, 0);
    } else {
        return bk_codes<QT_Q4_0>(mg, BkRaw{x, x >> 4, 0}, 0);
    }
}

template <int QT, int MT, int NW>
__global__ __launch_bounds__(64 * kBkWaves)
void k_gemm_block_staged(const uint8_t* __restrict__ W, const uint8_t* __restrict__ Waux,
                         const uint16_t* __restrict__ A, int lda, void* __restrict__ C, int ldc, int out_f16, int M,
                         int N, int K, int mcs) {
    constexpr int KS = kBkWaves / NW;                  // parts of K, each with NW waves and stages of its own
    constexpr int kStage = kStBlocks * MT * 1024;      // [block][row][lane row g] 16 bytes
    constexpr int kPieces = kStBlocks * MT * 64;   // 16-byte pieces of a step
    constexpr int PT = (kPieces + 64 * NW - 1) / (64 * NW);              // and per thread
    __shared__ __attribute__((aligned(16))) uint8_t all[KS * 2 * kStage];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int kg = __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * NW)), tid = (int)threadIdx.x - 64 * NW * kg;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t* const lds = all + kg * 2 * kStage;
    // workgroup u runs on XCD u % 8: each XCD gets a contiguous run of units,
    // the batch chunks of the same weight rows next to each other
    const int n_units = (int)gridDim.x, xcd = (int)blockIdx.x & 7, q8 = n_units >> 3, rem8 = n_units & 7;
    const int unit = xcd * q8 + min(xcd, rem8) + ((int)blockIdx.x >> 3);
    const int nc = unit / mcs, m0 = 16 * MT * (unit - nc * mcs);
    const int64_t nw = 16 * (NW * (int64_t)nc + wave) + r;         // this lane's weight row (output column)
    // this group's steps; what they hold past the last block counts as zero
    const int blocks = K >> 5, steps = (blocks + KS * kStBlocks - 1) / (KS * kStBlocks);
    const int first = kg * steps * kStBlocks;
    const int64_t n = min(nw, (int64_t)N - 1);
    const uint8_t* const row = W + n * (QT == QT_Q4_0 ? 18 * (int64_t)blocks : 16 * (int64_t)blocks);
    const uint8_t* const aux = QT == QT_Q4_0 ? nullptr : Waux + 2 * n * blocks;
    // piece f of a step: row f / 16, block f / 4 % 4, eight k from 8 (f % 4)
    const int pu = (tid >> 2) & 3, pp = tid & 3;
    const uint16_t* src[PT];
    uint32_t dst[PT];
    bool own[PT];
#pragma unroll
    for (int i = 0; i < PT; i++) {
        const int m = (tid >> 4) + 4 * NW * i;
        own[i] = m < 16 * MT;
        src[i] = A + (int64_t)min(m0 + m, M - 1) * lda + 8 * pp;
        dst[i] = (uint32_t)(pu * MT * 1024 + m * 64 + (QT == QT_PLANES ? 16 * pp : 32 * (pp & 1) + 8 * (pp >> 1)));
    }
    const Magic mg = make_magic();
    f4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) acc[i] = f4{0.f, 0.f, 0.f, 0.f};

    // loads without a branch (it would drain them all): past the last block they
    // read it again, and zeros are stored
    auto load_a = [&](B16a2 (&a)[PT], int s) {
        const int64_t k = 32 * (int64_t)min(first + kStBlocks * s + pu, blocks - 1);
#pragma unroll
        for (int i = 0; i < PT; i++) a[i] = *(const B16a2*)(src[i] + k);
    };
    auto store_a = [&](const B16a2 (&a)[PT], int s) {
        uint8_t* const st = lds + (s & 1) * kStage;
        const uint32_t on = first + kStBlocks * s + pu < blocks ? ~0u : 0u;
#pragma unroll
        for (int i = 0; i < PT; i++) {
            if (!own[i]) continue;
            if constexpr (QT == QT_PLANES) {
                *(u4*)(st + dst[i]) = u4{a[i].x & on, a[i].y & on, a[i].z & on, a[i].w & on};
            } else {
                *(uint2*)(st + dst[i]) = uint2{a[i].x & on, a[i].y & on};
                *(uint2*)(st + dst[i] + 16) = uint2{a[i].z & on, a[i].w & on};
            }
        }
    };
    // blocks past the last: its codes (finite) with a scale of zero
    auto load_w = [&](StRaw& w, int s) {
        w = st_load<QT>(row, aux, min(first + kStBlocks * s + g, blocks - 1));
    };

    B16a2 a[kStAhead][PT];
    StRaw w[kStAhead];
#pragma unroll
    for (int j = 0; j < kStAhead; j++) {
        load_w(w[j], j);
        load_a(a[j], j);
    }
    store_a(a[0], 0);
    load_a(a[0], kStAhead);
    barrier_lds();
    for (int s0 = 0; s0 < steps; s0 += kStAhead)
#pragma unroll
        for (int j = 0; j < kStAhead; j++) {
            const int s = s0 + j;
            if (s >= steps) break;
            float d[kStBlocks];
            uint32_t x[kStBlocks];
            if (first + kStBlocks * s + g >= blocks) w[j].d = 0;   // (its codes are finite)
            st_spread(w[j], x, d);
            load_w(w[j], s + kStAhead);
            store_a(a[(j + 1) % kStAhead], s + 1);
            load_a(a[(j + 1) % kStAhead], s + 1 + kStAhead);
            const uint8_t* const st = lds + (j & 1) * kStage + 64 * r + 16 * g;
#pragma unroll
            for (int u = 0; u < kStBlocks; u++) {
                const h8 q = st_codes<QT>(mg, x[u]);
                f4 p[MT];
#pragma unroll
                for (int i = 0; i < MT; i++)
                    p[i] = mfma16x16x32(*(const h8*)(st + (u * MT + i) * 1024), q, f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[i][e] = __builtin_fmaf(d[u], p[i][e], acc[i][e]);
            }
            barrier_lds();
        }
    if constexpr (KS == 2) {
        // group 1's sums to group 0 (the last step's barrier freed the stages)
        static_assert(KS * 2 * kStage >= NW * MT * 1024, "the hand-over fits the stages");
        f4* const hand = (f4*)all + wave * MT * 64 + lane;
        if (kg)
#pragma unroll
            for (int i = 0; i < MT; i++) hand[64 * i] = acc[i];
        __syncthreads();
        if (kg) return;
#pragma unroll
        for (int i = 0; i < MT; i++) acc[i] += hand[64 * i];
    }
    if (nw >= N) return;
    bool inf = false;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            inf |= __builtin_isinf(acc[i][e]);
            const int m = m0 + 16 * i + 4 * g + e;
            if (m >= M) break;
            store_out(acc[i][e], C, (int64_t)m * ldc + nw, out_f16);
        }
    if (inf)
        add_infinite_scales<QT>(4 * MT, [&](int x) { return m0 + 16 * (x >> 2) + 4 * g + (x & 3); }, W, Waux, A, lda, C,
                                ldc, out_f16, M, nw, blocks);
}

BlockPlan plan_of(const GemmArgs& g) {
    return plan_block(g.M, g.N, g.K, device_cus() > 0 ? device_cus() : 256);
}

template <int QT, int MT>
hipError_t launch_block(const GemmArgs& g, const BlockPlan& p, hipStream_t st) {
    if constexpr (MT >= 3) if (p.NT == 0) {            // (33 rows are three tiles)
        auto ks = p.NW == 8 ? k_gemm_block_staged<QT, MT, 8> : k_gemm_block_staged<QT, MT, 4>;
        hipLaunchKernelGGL(ks, dim3((unsigned)p.grid), dim3(64 * kBkWaves), 0, st, g.W, g.Waux, g.A, g.lda, g.C, g.ldc,
                           g.out_f16, g.M, g.N, g.K, p.nb);
        return hipGetLastError();
    }
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
    return (g.qtype == QT_Q4_0 || g.qtype == QT_PLANES) && g.K % 32 == 0 && !block_slower(g.M, g.N, g.K) &&
           launch_fits(plan_of(g).grid, 64 * kBkWaves);
}

hipError_t gemm_block(const GemmArgs& g, hipStream_t st) {
    const BlockPlan p = plan_of(g);
    return g.qtype == QT_Q4_0 ? dispatch_block<QT_Q4_0>(g, p, st) : dispatch_block<QT_PLANES>(g, p, st);
}

}  // namespace bf
