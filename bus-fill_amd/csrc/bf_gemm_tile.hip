// Tiled MFMA GEMM for prefill batches (more than 128 rows): k_gemm_tile.
//
//   C[m][n] = sum_k A[m][k] * dequant(W)[n][k]      (fp32 accumulation)
//
// Above 128 rows the dense kernel runs one launch per 128 rows, and each of
// them streams and decodes every weight again (17408 x 5120 at 2000 rows:
// 16 launches, 609-648 us, 545-585 TFLOP/s).  Here a workgroup computes a tile
// of up to 256 batch rows x 256 weight rows, K in steps of 64: both operands
// of a step sit in LDS as fp16, so a weight is decoded once per 256 rows and
// read from LDS by the waves of every column of the tile.
//
// * Eight waves, two per SIMD, 32 TA x 64 outputs each (TA x 2 tiles of
//   v_mfma_f32_32x32x16_f16: TA + 2 LDS reads feed 2 TA MFMAs).  NB = 2: 2 x 4
//   waves over a 256 x 256 tile.  NB = 1: 2 x 2 waves over a 64 TA x 128 tile,
//   twice, each set multiplying half of every step (their sums meet in LDS at
//   the end): the same reads per MFMA where 256 x 256 tiles leave CUs idle.
// * Activations: direct-to-LDS loads, one or two steps ahead (NS stages).
//   Weights: the quantized words in registers, loaded one super-group (four
//   steps) ahead, decoded to fp16 and written to the next step's stage.
// * One barrier per step.  A slot's fragments (16 k) are read from LDS while
//   the previous slot's multiply, across the barrier too, so the MFMAs never
//   wait for the LDS reads they use; the DMA instructions and the decode are
//   spread between the MFMAs, for one wave's issue stalls beside the other's
//   MFMAs (all of a step's DMA at its start: 388 us where spread takes 356,
//   2048 x 16384 x 5120).
// * LDS rows are 128 bytes (64 k); their 16-byte chunk c sits at c ^ ((row / 2)
//   % 8), so the 32 rows of a fragment read fall on distinct banks.
// * Bound by neither the matrix cores' rate nor the clock alone: MFMAs take
//   57-61 % of the SIMD cycles at 1.6-1.7 GHz with NB = 2 (2048 x 16384 x 5120:
//   328-336 us, 1020-1050 TFLOP/s) and 43-47 % at 1.9-2.0 GHz with NB = 1 (512 x
//   16384 x 5120: 93-97 us); an 8192^3 bf16 library product reached 1211 TFLOP/s on
//   such a chip, a library fp16 product of the first size takes 386-395 us on
//   decoded weights.  The compiler's own waits for the weight words count the DMAs
//   too (vmcnt(3) to vmcnt(6) once per step; planes, whose scales are copied while
//   fresh, vmcnt(0) once per super-group): stricter than the data needs, and not
//   yet taken out.  NB = 2 halves the operand traffic per flop of NB = 1 (2048
//   rows: 356 -> 327-340 us).
// * Measured (Q4_K, us per GEMM, before -> after): 17408 x 5120 at 512 / 2000
//   rows 150-165 / 609-648 -> 108 / 355-369; 5120 x 17408 at 2000 rows
//   572-606 -> 348-359; 5120 x 5120 at 300 / 512 rows 52-58 / 76-80 -> 35 / 43.
#include <atomic>

#include "bf_launch.h"
#include "bf_lds.h"
#include "bf_tile_plan.h"

namespace bf {
namespace {

struct __attribute__((packed, aligned(2))) U2a2 { uint32_t x, y; };
struct __attribute__((packed, aligned(2))) U4a2 { uint32_t x, y, z, w; };

// One thread's share of a super-group of its weight row: 4 / NB threads share
// a row (NB = 1: four, 8 code bytes of each 64-weight step; NB = 2: two, 16
// bytes), part j of each of the four steps, and the row's scales.  The code
// words of a step are reloaded for the next super-group as soon as they are
// decoded, so every load has four steps to arrive.
template <int NB> struct Codes { uint32_t w[2 * NB]; };
template <int QT, int NB> struct TileRaw;
template <int NB> struct TileRaw<QT_Q4_K, NB> { u4 hdr; Codes<NB> q[4]; };
template <int NB> struct TileRaw<QT_PLANES, NB> { u4 hdr; Codes<NB> q[4]; };
template <int NB> struct TileRaw<QT_Q4_0, NB> { uint32_t d[4]; Codes<NB> q[4]; };
template <int QT> constexpr int kStepLoads = QT == QT_Q4_0 ? 2 : 1;   // load instructions of a step's words
template <int QT> constexpr int kHdrLoads = QT == QT_Q4_0 ? 0 : 1;    // of the super-group's scales

template <int NB>
__device__ __forceinline__ void load_codes(Codes<NB>& c, const uint8_t* p) {
    if constexpr (NB == 1) {
        const U2a2 v = *(const U2a2*)p;
        c.w[0] = v.x; c.w[1] = v.y;
    } else {
        const U4a2 v = *(const U4a2*)p;
        c.w[0] = v.x; c.w[1] = v.y; c.w[2] = v.z; c.w[3] = v.w;
    }
}
// row: the row's first byte (planes: of the code plane; aux of the scale plane)
template <int QT, int NB>
__device__ __forceinline__ void load_step(TileRaw<QT, NB>& r, const uint8_t* row, int sg, int c, int j) {
    if constexpr (QT == QT_Q4_K) {
        load_codes<NB>(r.q[c], row + 144 * sg + 16 + 32 * c + 8 * NB * j);
    } else if constexpr (QT == QT_PLANES) {
        load_codes<NB>(r.q[c], row + 128 * sg + 32 * c + 8 * NB * j);
    } else {
        const uint8_t* p = row + 144 * sg + 36 * c + 18 * (NB == 1 ? j >> 1 : j);   // the block
        r.d[c] = *(const uint16_t*)p;
        load_codes<NB>(r.q[c], p + 2 + (NB == 1 ? 8 * (j & 1) : 0));
    }
}
template <int QT, int NB>
__device__ __forceinline__ void load_hdr(TileRaw<QT, NB>& r, const uint8_t* row, const uint8_t* aux, int sg) {
    if constexpr (QT == QT_Q4_K) r.hdr = *(const u4*)(row + 144 * sg);
    if constexpr (QT == QT_PLANES) r.hdr = ld16_a4(aux + 16 * sg);
}

// Scales of a super-group.  Q4_K: thread j of a row derives those of steps
// NB j .. NB j + NB - 1; step c takes them from its lane by DPP.
template <int QT, int NB> struct TileScl { u4 d; };
template <int NB> struct TileScl<QT_Q4_K, NB> { Scl<QT_Q4_K> s[NB]; };
template <int QT, int NB>
__device__ __forceinline__ void tile_scales(TileScl<QT, NB>& o, const TileRaw<QT, NB>& r, int j) {
    if constexpr (QT == QT_Q4_K) {
        Raw<QT_Q4_K> raw;
        raw.hdr = r.hdr;
#pragma unroll
        for (int i = 0; i < NB; i++) o.s[i] = scales(raw, NB * j + i);
    } else if constexpr (QT == QT_PLANES) {
        o.d = r.hdr;
    }
}
// lane C of the quad (NB = 1) or lane C of the lane pair (NB = 2)
template <int NB, int C>
__device__ __forceinline__ float row_lane(float v) {
    constexpr int ctrl = NB == 1 ? C * 0x55 : C | (C << 2) | ((2 + C) << 4) | ((2 + C) << 6);
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), ctrl, 0xF, 0xF, true));
}

// Piece I (0 .. 2 NB - 1) of a thread's 16 NB weights of step C: eight weights,
// k chunk tile_chunk(j, I) of the step.
template <int QT, int NB, int C, int I>
__device__ __forceinline__ h8 tile_decode(const Magic& mg, const TileRaw<QT, NB>& r, const TileScl<QT, NB>& s, int j) {
    if constexpr (QT == QT_PLANES) {
        return decode8_planes(mg, r.q[C].w[I], splat((s.d[C] >> (16 * (NB == 1 ? j >> 1 : j))) & 0xFFFFu));
    } else {
        constexpr bool HI = I >= NB;
        constexpr int w = 2 * (I % NB);
        if constexpr (QT == QT_Q4_0) {
            return decode8_q4_0<HI>(mg, r.q[C].w[w], r.q[C].w[w + 1], splat(r.d[C]));
        } else {
            const Scl<QT_Q4_K>& x = s.s[C % NB];
            constexpr int L = C / NB;
            return decode8_mix<HI>(r.q[C].w[w], r.q[C].w[w + 1], row_lane<NB, L>(HI ? x.sb : x.sa),
                                   row_lane<NB, L>(HI ? x.cb : x.ca));
        }
    }
}
template <int QT, int NB>
__host__ __device__ constexpr int tile_chunk(int j, int i) {
    if (QT == QT_PLANES) return 2 * NB * j + i;
    const int hi = i / NB, lo = i % NB;
    if (QT == QT_Q4_K) return NB * j + lo + 4 * hi;
    return NB == 1 ? 4 * (j >> 1) + (j & 1) + 2 * hi : 4 * j + lo + 2 * hi;
}

// Lane l copies 16 bytes from byte voff + soff of the buffer to LDS byte
// address m0 + 16 l.
__device__ __forceinline__ void dma16_buf(u4 rsrc, uint32_t voff, uint32_t soff, uint32_t m0) {
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" :: "v"(voff), "s"(rsrc), "s"(soff), "{m0}"(m0)
                 : "memory");
}

template <int V>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(V) : "memory");
}
// End of a phase: this wave's LDS traffic is done, and nothing moves across.
__device__ __forceinline__ void phase_end() {
    __builtin_amdgcn_sched_barrier(0);
    barrier_lds();
    __builtin_amdgcn_sched_barrier(0);
}

// Launch order -> unit: workgroup u runs on XCD u % 8, so each XCD gets a
// contiguous run of the n units (neighbouring units share operand panels, and
// each XCD has an L2 of its own).
__device__ __forceinline__ int xcd_unit(int u, int n) {
    const int x = u & 7, i = u >> 3, q = n >> 3, rem = n & 7;
    return x * q + min(x, rem) + i;
}

// x ^= D in place, where it is written (kept out of loop-invariant hoisting).
template <int D>
__device__ __forceinline__ void step_bits(uint32_t& x) {
    asm volatile("v_xor_b32 %0, %1, %0" : "+v"(x) : "n"(D));
}

// Tile index -> (m, n) tile: bands of kTlBand m-tiles, each n-tile by n-tile
// (the 32 tiles an XCD runs at once then share 4 + 8 operand panels; 1 % over
// m-tiles alone).
constexpr int kTlBand = 4;
__device__ __forceinline__ void tile_at(int tile, int mt, int nt, int& mi, int& ni) {
    const int b = tile / (kTlBand * nt), r = tile - b * kTlBand * nt, h = min(kTlBand, mt - b * kTlBand);
    ni = r / h;
    mi = b * kTlBand + r - ni * h;
}

// A tile of 64 TA batch rows x 128 NB weight rows.  NB = 2: 2 x 4 waves, each
// 32 TA x 64 outputs and the whole step.  NB = 1: 2 x 2 waves of the same size,
// twice (k groups 0 and 1: half of every step each, summed at the end).
template <int QT, int TA, int NB>
struct Tile {
    static constexpr int BM = 64 * TA, BN = 128 * NB, kAStage = BM * 128, kStage = kAStage + BN * 128;
    static constexpr int NS = NB == 1 ? 3 : 2;         // LDS stages
    static constexpr int KH = 2 * NB;                  // k16 slots of a step that a wave multiplies
    static constexpr int NP = 2 * NB;                  // decoded pieces of a thread and step
    static_assert(NS == 3 || kStage == 65536, "two stages differ in one address bit");

    u4 rsrc;
    uint32_t voff[TA];                   // activation DMA offsets
    uint32_t lds0;
    const uint8_t *row, *aux;
    int j, wave, last;
    // LDS bytes in a stage of this thread's first decoded piece and of the wave's
    // fragments of its first k16 slot; the other pieces and slots differ from
    // them in chunk bits only.  With two stages (64 KB apart) they walk through
    // pieces, slots and stages in place.
    uint32_t wst, fa, fw;
    Magic mg;
    TileRaw<QT, NB> raw;
    TileScl<QT, NB> scl;
    f16x acc[TA][2];
    h8 fa_[2][TA], fw_[2][2];

    __device__ __forceinline__ uint32_t piece(int i) const { return wst ^ (16u * tile_chunk<QT, NB>(0, i)); }
    // piece q of a step's activations
    __device__ __forceinline__ void dma(int q, int step, uint32_t stage) {
        dma16_buf(rsrc, voff[q], 128u * (uint32_t)step, lds0 + stage + 1024u * (uint32_t)(wave + 8 * q));
    }
    // Slot H of a step: its fragments are read from stage st while the previous
    // slot's multiply.
    template <int H>
    __device__ __forceinline__ void read(const uint8_t* lds, uint32_t st) {
        if constexpr (NS == 2) {
            step_bits<32 * (H ^ ((H + KH - 1) % KH)) | (H == 0 ? kStage : 0)>(fa);
            step_bits<32 * (H ^ ((H + KH - 1) % KH)) | (H == 0 ? kStage : 0)>(fw);
        }
        const uint32_t xa = NS == 2 ? fa : (fa ^ (32 * H)) + st, xw = NS == 2 ? fw : (fw ^ (32 * H)) + st;
#pragma unroll
        for (int b = 0; b < 2; b++) fw_[H & 1][b] = *(const h8*)(lds + xw + 4096 * b);
#pragma unroll
        for (int t = 0; t < TA; t++) fa_[H & 1][t] = *(const h8*)(lds + xa + 4096 * t);
    }
    template <int P>
    __device__ __forceinline__ void mma(int t0, int t1) {
#pragma unroll
        for (int t = t0; t < t1; t++)
#pragma unroll
            for (int b = 0; b < 2; b++) acc[t][b] = mfma32x32x16(fa_[P][t], fw_[P][b], acc[t][b]);
    }
    template <int H, int C, bool DEC, bool DMA, bool RELOAD>
    __device__ __forceinline__ void slot(uint8_t* lds, int sg, uint32_t st0, uint32_t st1, uint32_t std) {
        constexpr int TH = (TA + 1) / 2, D = (C + 1) & 3;
        const int ds = 4 * sg + C + NS - 1;
        h8 o;
        if constexpr (DMA && 2 * H < TA) dma(2 * H, ds, std);
        read<H>(lds, st0);
        mma<(H + 1) & 1>(0, TH);
        if constexpr (DEC) o = tile_decode<QT, NB, D, H>(mg, raw, scl, j);
        if constexpr (DMA && 2 * H + 1 < TA) dma(2 * H + 1, ds, std);
        if constexpr (RELOAD && H == KH - 1) {
            // the step's words are decoded: the next super-group's into their place
            load_step<QT, NB>(raw, row, C < 3 ? sg + 1 : min(sg + 2, last), D, j);
            if constexpr (C == 3) load_hdr<QT, NB>(raw, row, aux, min(sg + 2, last));
        }
        mma<(H + 1) & 1>(TH, TA);
        if constexpr (DEC) {
            if constexpr (NS == 2) {
                constexpr int P = (H + NP - 1) % NP;
                step_bits<16 * (tile_chunk<QT, NB>(0, H) ^ tile_chunk<QT, NB>(0, P)) | (H == 0 ? kStage : 0)>(wst);
                *(h8*)(lds + wst) = o;
            } else {
                *(h8*)(lds + piece(H) + st1) = o;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // Step C of super-group sg (LAST: the range's last one): multiplies stage
    // st0 (its last slot in the next step), decodes the next step's weights
    // into st1 and starts the activations NS - 1 steps ahead.
    template <int C, bool LAST>
    __device__ __forceinline__ void step(uint8_t* lds, int sg, uint32_t* st) {
        constexpr bool kDec = !(LAST && C == 3), kDma = !(LAST && C >= 5 - NS);
        constexpr int n0 = LAST ? 0 : kStepLoads<QT> + (C == 3 ? kHdrLoads<QT> : 0);     // this step's reloads
        constexpr int n1 = C == 0 ? kStepLoads<QT> + kHdrLoads<QT> : LAST ? 0 : kStepLoads<QT>;   // the previous step's
        // two stages alternate (a range starts on stage 0), three rotate
        const uint32_t x0 = NS == 2 ? (C & 1) * kStage : st[0], x1 = NS == 2 ? (1 - (C & 1)) * kStage : st[1];
        const uint32_t xd = NS == 2 ? x1 : st[NS - 1];
        if constexpr (!LAST && C == 3) tile_scales<QT, NB>(scl, raw, j);
        slot<0, C, kDec, kDma, !LAST>(lds, sg, x0, x1, xd);
        slot<1, C, kDec, kDma, !LAST>(lds, sg, x0, x1, xd);
        if constexpr (KH > 2) {
            slot<2, C, kDec, kDma, !LAST>(lds, sg, x0, x1, xd);
            slot<3, C, kDec, kDma, !LAST>(lds, sg, x0, x1, xd);
        }
        // the next step's activations have landed when at most the loads issued
        // after them are outstanding
        if constexpr (NS == 2) wait_vm<n0>();
        else wait_vm<kDma ? TA + n0 + n1 : 0>();
        phase_end();
        if constexpr (NS == 3) {
            const uint32_t t = st[0];
            st[0] = st[1];
            st[1] = st[2];
            st[2] = t;
        }
    }
    __device__ __forceinline__ void run(uint8_t* lds, int s0, int s1) {
        uint32_t st[NS];
#pragma unroll
        for (int i = 0; i < NS; i++) st[i] = i * kStage;
        last = s1 - 1;
        load_hdr<QT, NB>(raw, row, aux, s0);
#pragma unroll
        for (int c = 0; c < 4; c++) load_step<QT, NB>(raw, row, s0, c, j);
#pragma unroll
        for (int q = 0; q < TA; q++) dma(q, 4 * s0, st[0]);
        if constexpr (NS == 3) {
#pragma unroll
            for (int q = 0; q < TA; q++) dma(q, 4 * s0 + 1, st[1]);
        }
        tile_scales<QT, NB>(scl, raw, j);
        *(h8*)(lds + piece(0)) = tile_decode<QT, NB, 0, 0>(mg, raw, scl, j);
        *(h8*)(lds + piece(1)) = tile_decode<QT, NB, 0, 1>(mg, raw, scl, j);
        if constexpr (NP > 2) {
            *(h8*)(lds + piece(2)) = tile_decode<QT, NB, 0, 2 % NP>(mg, raw, scl, j);
            *(h8*)(lds + piece(3)) = tile_decode<QT, NB, 0, 3 % NP>(mg, raw, scl, j);
        }
        load_step<QT, NB>(raw, row, min(s0 + 1, last), 0, j);
        load_hdr<QT, NB>(raw, row, aux, min(s0 + 1, last));
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int e = 0; e < 8; e++) fw_[1][b][e] = 0;
#pragma unroll
        for (int t = 0; t < TA; t++)
#pragma unroll
            for (int e = 0; e < 8; e++) fa_[1][t][e] = 0;
        wait_vm<(NS - 2) * TA + kStepLoads<QT> + kHdrLoads<QT>>();
        phase_end();
        if constexpr (NS == 2) {                       // where the previous step would have left them
            fa ^= 32 * (KH - 1) | kStage;
            fw ^= 32 * (KH - 1) | kStage;
            wst = piece(NP - 1);
        }
        int sg = s0;
        for (; sg < last; sg++) {
            step<0, false>(lds, sg, st);
            step<1, false>(lds, sg, st);
            step<2, false>(lds, sg, st);
            step<3, false>(lds, sg, st);
        }
        step<0, true>(lds, sg, st);
        step<1, true>(lds, sg, st);
        step<2, true>(lds, sg, st);
        step<3, true>(lds, sg, st);
        mma<1>(0, TA);
    }
};

// Workgroups [0, F): whole tiles, straight to C.  Workgroups F ..: the R =
// tiles - F remaining ones, each cut in S ranges of super-groups whose sums go
// to the workspace ([split][tile][row][128 NB] fp32; S > 1) for k_tile_sum.
template <int QT, int TA, int NB>
__global__ __launch_bounds__(kTlThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_gemm_tile(const uint8_t* W, const uint8_t* Waux, const uint16_t* A, int lda, void* C, int ldc, int out_f16,
                 int M, int N, int K, int mt, int F, int R, int S, float* ws) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    using T = Tile<QT, TA, NB>;
    constexpr int BM = T::BM, BN = T::BN;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nsg = K >> 8;
    int tile, sp = 0, s0 = 0, s1 = nsg;
    if ((int)blockIdx.x < F) {
        tile = xcd_unit((int)blockIdx.x, F);
    } else {
        const int v = xcd_unit((int)blockIdx.x - F, R * S);
        sp = v / R;
        tile = F + v - sp * R;
        s0 = sp * nsg / S;
        s1 = (sp + 1) * nsg / S;
    }
    int mi, ni;
    tile_at(tile, mt, (N + BN - 1) / BN, mi, ni);
    const int m0 = mi * BM, n0 = ni * BN;
    const int rows = min(BM, M - m0);

    T t;
    const uint16_t* const a0 = A + (int64_t)m0 * lda;
    t.rsrc = u4{(uint32_t)(uintptr_t)a0, (uint32_t)((uintptr_t)a0 >> 32) & 0xFFFFu,
                (uint32_t)(((int64_t)(rows - 1) * lda + K) * 2), 0x00020000u};
#pragma unroll
    for (int q = 0; q < TA; q++) {
        const int r = min(8 * (wave + 8 * q) + (lane >> 3), rows - 1);
        t.voff[q] = (uint32_t)r * (uint32_t)lda * 2u + 16u * (((uint32_t)lane & 7u) ^ (4u * (wave & 1) + (lane >> 4)));
    }
    t.lds0 = lds_addr(lds);
    t.wave = wave;
    constexpr int TPR = 4 / NB;                        // threads of a weight row
    t.j = threadIdx.x % TPR;
    const int wr = threadIdx.x / TPR;
    const int64_t n = min(n0 + wr, N - 1);
    t.row = W + n * row_bytes(QT, K);
    t.aux = QT == QT_PLANES ? Waux + n * (K >> 4) : nullptr;
    t.wst = T::kAStage + wr * 128 + 16 * (tile_chunk<QT, NB>(t.j, 0) ^ ((wr >> 1) & 7));
    const int kg = NB == 1 ? wave >> 2 : 0, wm = NB == 1 ? (wave >> 1) & 1 : wave >> 2, wn = wave & (2 * NB - 1);
    const uint32_t f = (lane & 31) * 128 + 16 * ((4 * kg + (lane >> 5)) ^ ((lane >> 1) & 7));
    t.fa = wm * (32 * TA * 128) + f;
    t.fw = T::kAStage + wn * (64 * 128) + f;
    t.mg = make_magic();
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int e = 0; e < 16; e++) t.acc[a][b][e] = 0.f;
    t.run(lds, s0, s1);

    // Outputs of the wave: rows mr + (8 (e / 4) + e % 4) of every 32-row tile,
    // column nn (+ 32 b).
    const int nc = n0 + 64 * wn + (lane & 31), mr = 32 * TA * wm + 4 * (lane >> 5);
    const bool part = (int)blockIdx.x >= F && S > 1;
    float* const pw = ws + (size_t)(sp * R + tile - F) * (BM * BN) + (size_t)mr * BN + (nc - n0);
    auto store = [&](int dm, int b, float y) {
        const int m = m0 + mr + dm, nn = nc + 32 * b;
        if (m >= M) return;
        if (part) {
            pw[(size_t)dm * BN + 32 * b] = y;
        } else if (nn < N) {
            const int64_t o = (int64_t)m * ldc + nn;
            if (out_f16) ((_Float16*)C)[o] = (_Float16)y;
            else ((float*)C)[o] = y;
        }
    };
    if constexpr (NB == 2) {
#pragma unroll
        for (int a = 0; a < TA; a++)
#pragma unroll
            for (int e = 0; e < 16; e++)
#pragma unroll
                for (int b = 0; b < 2; b++) store(32 * a + 8 * (e / 4) + e % 4, b, t.acc[a][b][e]);
    } else {
        // The two k groups' sums: wave (kg, wm, wn) hands the column tile 1 - kg
        // to its partner and finishes column tile kg.
        uint8_t* const xch = lds + (threadIdx.x & 255) * 16;
        constexpr int XB = TA * 4 * 4096;              // bytes handed over by one k group
#pragma unroll
        for (int a = 0; a < TA; a++)
#pragma unroll
            for (int e = 0; e < 16; e += 4) {
                const f16x& v = kg ? t.acc[a][0] : t.acc[a][1];
                *(f4*)(xch + kg * XB + (a * 4 + e / 4) * 4096) = f4{v[e], v[e + 1], v[e + 2], v[e + 3]};
            }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < TA; a++)
#pragma unroll
            for (int e = 0; e < 16; e += 4) {
                const f4 x = *(const f4*)(xch + (1 - kg) * XB + (a * 4 + e / 4) * 4096);
                const f16x& v = kg ? t.acc[a][1] : t.acc[a][0];
#pragma unroll
                for (int i = 0; i < 4; i++) store(32 * a + 2 * e + i, kg, kg ? x[i] + v[e + i] : v[e + i] + x[i]);
            }
    }
}

// C of the cut tiles: their S partial sums in split order.  Block (r, y):
// 1024 / BN rows of the r-th cut tile, four columns per thread.
template <int BM, int BN>
__global__ __launch_bounds__(256) void k_tile_sum(const float* __restrict__ ws, void* __restrict__ C, int ldc,
                                                  int out_f16, int M, int N, int mt, int F, int R, int S) {
    constexpr int Q = BN / 4;                          // column quads of a row
    const int r = (int)blockIdx.x, tile = F + r;
    int mi, ni;
    tile_at(tile, mt, (N + BN - 1) / BN, mi, ni);
    const int dm = 256 / Q * (int)blockIdx.y + (int)threadIdx.x / Q, m = mi * BM + dm, nl = 4 * ((int)threadIdx.x % Q);
    if (m >= M) return;
    const float* p = ws + (size_t)r * (BM * BN) + (size_t)dm * BN + nl;
    const size_t ps = (size_t)R * (BM * BN);
    f4 s = f4{0.f, 0.f, 0.f, 0.f};
    for (int q0 = 0; q0 < S; q0 += 8) {
        f4 x[8];
#pragma unroll
        for (int k = 0; k < 8; k++) x[k] = q0 + k < S ? *(const f4*)(p + (q0 + k) * ps) : f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (q0 + k < S) s += x[k];
    }
    const int64_t n0 = (int64_t)ni * BN + nl, o = (int64_t)m * ldc + n0;
    if (((uintptr_t)C & 15) == 0 && (ldc & 3) == 0 && n0 + 3 < N) {
        if (out_f16) {
            typedef _Float16 h4 __attribute__((ext_vector_type(4)));
            *(h4*)((_Float16*)C + o) = h4{(_Float16)s[0], (_Float16)s[1], (_Float16)s[2], (_Float16)s[3]};
        } else {
            *(f4*)((float*)C + o) = s;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (n0 + i >= N) break;
            if (out_f16) ((_Float16*)C)[o + i] = (_Float16)s[i];
            else ((float*)C)[o + i] = s[i];
        }
    }
}

bool plan_of(const GemmArgs& g, TilePlan& p) {
    if ((int64_t)g.lda >= (1 << 22)) return false;     // activation offsets of a tile in 32 bits
    // a caller's workspace of the size that 128-row launches of the dense kernel
    // take on this matrix serves here too
    GemmArgs slice = g;
    slice.M = 128;
    const size_t scratch = dense_supports(slice) ? dense_scratch_bytes(slice) : 0;
    return plan_tile(g.M, g.N, g.K, device_cus() > 0 ? device_cus() : 256, scratch, p);
}

template <int QT, int TA, int NB>
hipError_t launch_tile(const GemmArgs& g, const TilePlan& p, const Scratch* scratch, hipStream_t st) {
    using T = Tile<QT, TA, NB>;
    auto k = k_gemm_tile<QT, TA, NB>;
    constexpr int lds = T::NS * T::kStage;
    static std::atomic<uint64_t> attr_set{0};          // one bit per device: LDS limit raised
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (!(attr_set.load(std::memory_order_acquire) & bit)) {
        e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        attr_set.fetch_or(bit, std::memory_order_acq_rel);
    }
    unsigned* counters = nullptr;
    float* parts = nullptr;
    if (p.part) {
        e = split_workspace(scratch, st, 0, p.part, &counters, &parts);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k, dim3(p.F + p.R * p.S), dim3(kTlThreads), lds, st, g.W, g.Waux, g.A, g.lda, g.C, g.ldc,
                       g.out_f16, g.M, g.N, g.K, p.mt, p.F, p.R, p.S, parts);
    e = hipGetLastError();
    if (e != hipSuccess || !p.part) return e;
    hipLaunchKernelGGL((k_tile_sum<T::BM, T::BN>), dim3(p.R, T::BM * T::BN / 1024), dim3(256), 0, st, (const float*)parts,
                       g.C, g.ldc, g.out_f16, g.M, g.N, p.mt, p.F, p.R, p.S);
    return hipGetLastError();
}

template <int QT>
hipError_t dispatch_tile(const GemmArgs& g, const TilePlan& p, const Scratch* scratch, hipStream_t st) {
    if (p.NB == 2) return launch_tile<QT, 4, 2>(g, p, scratch, st);
    if (p.TA == 2) return launch_tile<QT, 2, 1>(g, p, scratch, st);
    if (p.TA == 3) return launch_tile<QT, 3, 1>(g, p, scratch, st);
    return launch_tile<QT, 4, 1>(g, p, scratch, st);
}

}  // namespace

bool tile_supports(const GemmArgs& g) {
    TilePlan p;
    if (!plan_of(g, p)) return false;
    GemmArgs slice = g;
    slice.M = 128;
    return !(dense_supports(slice) &&
             slices_faster(g.M, g.N, g.K, device_cus() > 0 ? device_cus() : 256,
                           g.qtype == QT_PLANES ? 1.12 : g.qtype == QT_Q4_0 ? 1.08 : 1.04, p));
}

size_t tile_scratch_bytes(const GemmArgs& g) {
    TilePlan p;
    return plan_of(g, p) ? p.part : 0;
}

WsNeed tile_ws_need(const GemmArgs& g) {
    WsNeed w;
    w.p = tile_scratch_bytes(g);
    return w;
}

hipError_t gemm_tile(const GemmArgs& g, const Scratch* scratch, hipStream_t st) {
    TilePlan p;
    if (!plan_of(g, p)) return hipErrorInvalidValue;
    if (g.qtype == QT_PLANES) return dispatch_tile<QT_PLANES>(g, p, scratch, st);
    if (g.qtype == QT_Q4_0) return dispatch_tile<QT_Q4_0>(g, p, scratch, st);
    return dispatch_tile<QT_Q4_K>(g, p, scratch, st);
}

}  // namespace bf
