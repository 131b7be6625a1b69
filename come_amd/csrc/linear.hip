// Linear layers: out = act(x W^T + b), x [rows, K], W [N, K], 16 bits in and out, fp32 accumulation (gfx950).
//
// A merged clip of a few frames has 200 - 5000 packed rows.  A product of that height is a round or two of workgroups, so what
// counts is how many CUs have a tile, how few bytes a tile moves from L2 to LDS per multiplication, and what stands in front
// of and behind its key loop.  On taller ones the product itself runs at the chip's power limit whoever computes it, and what
// is left to gain is the pass over memory that GELU costs as an operation of its own.
//
// A workgroup of QM x QN wavefronts computes a BM x BN tile of the output; K is walked in steps of 64.  Rows of x and W go
// global -> LDS by direct loads into a ring of S stages (the 16-byte chunks of a row permuted, so that fragment reads are
// free of bank conflicts), spread over the matrix instructions of a step; one barrier a step.  Fragments of a 32-wide k-step
// are read while the one before is multiplied.  Products are formed transposed, W x^T, so that a lane holds four consecutive
// outputs of one row; the accumulators start from the bias.  Results pass through LDS and leave as 16-byte stores.
// Every output is one chain of additions in the order of K, whatever the tile: its bits do not depend on the shape chosen.
//
// What bounds it, by variants of the loop that leave one part out (128 x 256, us a step of 64): matrix instructions alone 0.46,
// direct loads alone 0.45 (48 KiB: 49 of the 64 bytes a cycle that a CU's path from L2 moves), fragment reads alone 0.24, all
// together 0.52 with 78 workgroups and 0.71 with 208, which is 1230 TFLOP/s, what large products sustain as well; 4 - 5 us
// around the loop.  Two wavefronts per SIMD hide the issue of direct loads that one alone waits in (0.58 a step).
//
// v_mfma 16x16x32 and not 32x32x16: the clock of a busy chip follows the power it draws, and the former moves 8 registers of sums
// in and out for 16 cycles of the matrix pipe, the latter 32 for 32.  Full chip, N(0, 1) operands read from LDS, nothing else:
// 2500 and 2250 TFLOP/s.  us, 32x32x16 and 16x16x32: 1596 rows, qkv 15.1 and 14.9, fc1 with GELU 20.6 and 20.3,
// fc2 in shares 19.6 and 19.1; 800 rows 11.5 and 11.1, 14.5 and 13.8, 14.8 and 13.5; 25 536 rows, fc1 with GELU 246.8 and 242.7; a
// forward of two frames 6235 and 6145.
#include "attn_common.h"

#include <algorithm>
#include <cmath>

namespace come {
namespace {

struct LinearArgs {
    const char *x, *w;
    const uint16_t *bias;            // [N] or nullptr
    uint16_t *out;
    float *partial;                  // SPLIT: [splits][rows][N], sums without the bias
    int rows, K, N;
    int m_tiles, n_tiles, splits, per_xcd;
};

constexpr int kGroupN = 8;

// x Phi(x) with the erfc of Abramowitz and Stegun 7.1.26 (|error| <= 1.5e-7, relative to exp(-x^2 / 2) in the tail)
__device__ __forceinline__ float gelu(float x) {
    const float ax = fmaxf(-x, fminf(x, 100.f));                  // |x|; 100 for infinity, whose 1 - Phi is 0 (minus infinity gives NaN, as in torch)
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(ax, 0.3275911f * 0.70710678f, 1.0f));
    const float e = __builtin_amdgcn_exp2f(x * x * -0.72134752f);
    float p = __builtin_fmaf(t, 0.5f * 1.061405429f, 0.5f * -1.453152027f);
    p = __builtin_fmaf(p, t, 0.5f * 1.421413741f);
    p = __builtin_fmaf(p, t, 0.5f * -0.284496736f);
    p = __builtin_fmaf(p, t, 0.5f * 0.254829592f);
    const float q = p * t * e;                                    // 1 - Phi(|x|)
    return __builtin_fmaf(-ax, q, fmaxf(x, 0.f));
}

// SPLIT: a tile is computed by `splits` workgroups, each over its share of K; their sums meet in the kernel behind
// (come_residual_norm_split).
// `first`: workgroups of the launch in front of those of these tiles, a multiple of 8.
template <int BM, int BN, int S> constexpr int kTileBytes = S * (BM + BN) * 128;
template <int BN> constexpr int kTileBias = (BN + 127) / 128 * 128;
template <int DT, int BM, int BN, int QM, int QN, int S, int ACT, bool SPLIT>
__device__ __forceinline__ void linear_tile(const LinearArgs a, uint32_t first, char *lds, uint16_t *lds_bias) {
    using E = Elem<DT>;
    constexpr int WAVES = QM * QN, WM = BM / QM, WN = BN / QN, MT = WM / 16, NT = WN / 16;
    static_assert(WM % 32 == 0 && WN % 32 == 0, "results leave 32 rows at a time");
    constexpr int kStage = (BM + BN) * 128;                       // bytes
    constexpr int DX = BM / 8 / WAVES, DW = BN / 8 / WAVES, D = DX + DW;        // direct loads of a wavefront per step
    constexpr int kPitch = WN * 2 + 16;                           // bytes of a row of results in LDS
    static_assert(WAVES * 32 * (SPLIT ? 144 : kPitch) <= S * kStage, "the results fit the ring");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int wm = wave % QM, wn = wave / QM, r = lane & 15, g = lane >> 4;

    // Workgroup i runs on XCD i % 8, each with its own L2: an XCD takes a contiguous range of the tiles, which are counted row
    // by row within groups of kGroupN columns, so that its L2 holds few rows of x and of W at a time.  4096 -> 1024 with 1596 rows
    // 23.3 us in columns, 21.9 in groups of 8; 1024 -> 4096 with 25 536 rows 225 and 213 (groups of 4 - 16 are alike).
    const int local = static_cast<int>((blockIdx.x - first) >> 3), item = static_cast<int>(blockIdx.x & 7u) * a.per_xcd + local;
    const int tiles = a.m_tiles * a.n_tiles;
    if (local >= a.per_xcd || item >= tiles * (SPLIT ? a.splits : 1)) return;
    const int share = SPLIT ? __builtin_amdgcn_readfirstlane(item / tiles) : 0, lin = item - share * tiles;
    const int group = lin / (a.m_tiles * kGroupN), in_group = lin - group * (a.m_tiles * kGroupN);
    const int width = min(kGroupN, a.n_tiles - group * kGroupN);
    const int mt = __builtin_amdgcn_readfirstlane(in_group / width);
    const int nt = __builtin_amdgcn_readfirstlane(group * kGroupN + in_group - mt * width);
    const int m0 = mt * BM, n0 = nt * BN;
    const int K = a.K;
    const int k_first = SPLIT ? __builtin_amdgcn_readfirstlane(share * (K / 64) / a.splits) : 0;          // in steps
    const int steps = SPLIT ? __builtin_amdgcn_readfirstlane((share + 1) * (K / 64) / a.splits) - k_first : K / 64;
    const char *const x_tile = a.x + static_cast<int64_t>(m0) * K * 2 + k_first * 128, *const w_tile = a.w + static_cast<int64_t>(n0) * K * 2 + k_first * 128;
    uint32_t x_off[DX], w_off[DW];
    const uint32_t row_bytes = static_cast<uint32_t>(K) * 2u;
#pragma unroll
    for (int i = 0; i < DX; ++i) {
        const int row = (wave * DX + i) * 8 + (lane >> 3);
        x_off[i] = static_cast<uint32_t>(min(row, a.rows - 1 - m0)) * row_bytes + static_cast<uint32_t>((lane & 7) ^ ((row >> 1) & 7)) * 16u;
    }
#pragma unroll
    for (int i = 0; i < DW; ++i) {
        const int row = (wave * DW + i) * 8 + (lane >> 3);
        w_off[i] = static_cast<uint32_t>(min(row, a.N - 1 - n0)) * row_bytes + static_cast<uint32_t>((lane & 7) ^ ((row >> 1) & 7)) * 16u;
    }
    const uint32_t lds0 = lds_address(lds);
    int k_next = 0;                                               // step of K that is staged next
    uint32_t stage_in = 0;                                        // where to
    auto load = [&](int i) __attribute__((always_inline)) {       // direct load i of the step
        const int64_t at = static_cast<int64_t>(k_next) * 128;
        if (i < DX) dma_b128(x_tile + at, x_off[i], lds0 + stage_in + static_cast<uint32_t>((wave * DX + i) * 1024));
        else dma_b128(w_tile + at, w_off[i - DX], lds0 + stage_in + static_cast<uint32_t>(BM * 128 + (wave * DW + i - DX) * 1024));
    };
    auto staged = [&]() __attribute__((always_inline)) {
        ++k_next;
        stage_in = stage_in + kStage == S * kStage ? 0u : stage_in + kStage;
    };

    if (!SPLIT && a.bias != nullptr && wave < (BN + 127) / 128)
        dma_b32(reinterpret_cast<const char *>(a.bias), static_cast<uint32_t>(min(n0 + 128 * wave + 2 * lane, a.N - 2)) * 2u,
                lds_address(lds_bias + 128 * wave));
#pragma unroll
    for (int s = 0; s < S - 1; ++s) {
        if (s < steps) {
#pragma unroll
            for (int i = 0; i < D; ++i) load(i);
            staged();
        }
    }

    uint32_t rd[2];                                               // fragment k-step ks of row r: features 32 ks + 8 g .. + 7
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) rd[ks] = static_cast<uint32_t>(r * 128 + (((4 * ks + g) ^ ((r >> 1) & 7)) << 4));
    const char *const x_lds = lds + wm * WM * 128, *const w_lds = lds + BM * 128 + wn * WN * 128;
    u32x4 xf[2][MT], wf[2][NT];
    auto read = [&](int buf, uint32_t stage, int ks, int f) __attribute__((always_inline)) {      // fragment f of a k-step
        if (f < MT) xf[buf][f] = *reinterpret_cast<const u32x4 *>(x_lds + stage + rd[ks] + f * 2048);
        else wf[buf][f - MT] = *reinterpret_cast<const u32x4 *>(w_lds + stage + rd[ks] + (f - MT) * 2048);
    };
    if (steps >= S - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * D) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    uint32_t stage = 0;
#pragma unroll
    for (int f = 0; f < MT + NT; ++f) read(0, stage, 0, f);

    f32x4 acc[NT][MT];                                            // outputs 16 i + 4 g .. + 3 of row 16 j + r
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        f32x4 b = {0.f, 0.f, 0.f, 0.f};
        if (!SPLIT && a.bias != nullptr) {
            const u32x2 w = *reinterpret_cast<const u32x2 *>(lds_bias + wn * WN + 16 * i + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) b[e] = E::to_f32(static_cast<uint16_t>(e & 1 ? w[e >> 1] >> 16 : w[e >> 1] & 0xffffu));
        }
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = b;
    }
    constexpr int kPerStep = MT * NT;                             // matrix instructions of a k-step
    constexpr int kReads = kPerStep * 3 / 4;                      // the next k-step's fragments go out with the first of them
    for (int t = 0; t < steps; ++t) {
        const bool more = t + S - 1 < steps;
        const uint32_t next_stage = stage + kStage == S * kStage ? 0u : stage + kStage;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int cur = ks, nxt = ks ^ 1;
            if (ks == 1) {
                // this stage has been read, the next one has landed
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * D) : "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                asm volatile("s_barrier" ::: "memory");
            }
            int f = 0;
#pragma unroll
            for (int m = 0; m < kPerStep; ++m) {
                const int i = m / MT, j = m % MT;
                acc[i][j] = E::mfma16(wf[cur][i], xf[cur][j], acc[i][j]);
                __builtin_amdgcn_sched_barrier(0);
                const int want = ((m + 1) * (MT + NT) + kReads - 1) / kReads;
#pragma unroll
                for (; f < want && f < MT + NT; ++f)
                    if (ks == 0) read(nxt, stage, 1, f);
                    else read(nxt, next_stage, 0, f);
                if (ks == 0 && more) {                            // and the direct loads
#pragma unroll
                    for (int d = m * D / kPerStep; d < (m + 1) * D / kPerStep; ++d) load(d);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (more) staged();
        stage = next_stage;
    }

    // ---- results: 32 rows at a time through a part of LDS that is this wavefront's alone (16 bytes of padding a row), then
    // 16-byte stores
    __syncthreads();                                              // nobody reads the ring any more
    if constexpr (SPLIT) {                                        // 32 x 32 sums at a time, stored as rows of 128 bytes
        char *const mine = lds + wave * (32 * 144);
        float *const part = a.partial + static_cast<int64_t>(share) * a.rows * a.N;
#pragma unroll
        for (int j = 0; j < MT / 2; ++j)
#pragma unroll
            for (int i = 0; i < NT / 2; ++i) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<f32x4 *>(mine + (16 * (q >> 1) + r) * 144 + (16 * (q & 1) + 4 * g) * 4) = acc[2 * i + (q & 1)][2 * j + (q >> 1)];
                const int col = n0 + wn * WN + 32 * i + 4 * (lane & 7);
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const int row = m0 + wm * WM + 32 * j + 8 * p + (lane >> 3);
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(mine + (8 * p + (lane >> 3)) * 144 + (lane & 7) * 16);
                    if (row < a.rows && col < a.N) *reinterpret_cast<f32x4 *>(part + static_cast<int64_t>(row) * a.N + col) = v;
                }
            }
        return;
    }
    char *const mine = lds + wave * (32 * kPitch);
    constexpr int kChunks = WN / 8;                               // 16-byte chunks a row
    const int col0 = n0 + wn * WN;
#pragma unroll
    for (int j = 0; j < MT / 2; ++j) {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = ACT == COME_ACT_GELU ? gelu(acc[i][2 * j + q][e]) : acc[i][2 * j + q][e];
                *reinterpret_cast<u32x2 *>(mine + (16 * q + r) * kPitch + (16 * i + 4 * g) * 2) = u32x2{E::pack2(v[0], v[1]), E::pack2(v[2], v[3])};
            }
        const int row0 = m0 + wm * WM + 32 * j;
#pragma unroll
        for (int p = 0; p < 32 * kChunks / 64; ++p) {
            const int at = p * 64 + lane, row = at / kChunks, c = at % kChunks;
            const u32x4 v = *reinterpret_cast<const u32x4 *>(mine + row * kPitch + c * 16);
            if (row0 + row < a.rows && col0 + 8 * c < a.N) {
                u32x4 *const to = reinterpret_cast<u32x4 *>(a.out + static_cast<int64_t>(row0 + row) * a.N + col0 + 8 * c);
                __builtin_nontemporal_store(v, to);
            }
        }
    }
}

template <int DT, int BM, int BN, int QM, int QN, int S, int ACT, bool SPLIT>
__global__ __launch_bounds__(64 * QM * QN) void linear_kernel(const LinearArgs a) {
    __shared__ __attribute__((aligned(1024))) char lds[kTileBytes<BM, BN, S>];
    __shared__ __attribute__((aligned(256))) uint16_t lds_bias[kTileBias<BN>];
    linear_tile<DT, BM, BN, QM, QN, S, ACT, SPLIT>(a, 0, lds, lds_bias);
}

// Two parts of the rows in one launch, with GELU: `a` in 256 x 256 tiles, `b` in BM x BN (whole_rounds).
template <int DT, int BM, int BN, int QM, int QN, int S>
__global__ __launch_bounds__(512) void linear_mixed_kernel(const LinearArgs a, const LinearArgs b) {
    __shared__ __attribute__((aligned(1024))) char lds[std::max(kTileBytes<256, 256, 2>, kTileBytes<BM, BN, S>)];
    __shared__ __attribute__((aligned(256))) uint16_t lds_bias[kTileBias<256>];
    const uint32_t first = 8u * a.per_xcd;
    if (blockIdx.x < first) linear_tile<DT, 256, 256, 2, 4, 2, COME_ACT_GELU, false>(a, 0, lds, lds_bias);
    else linear_tile<DT, BM, BN, QM, QN, S, COME_ACT_GELU, false>(b, first, lds, lds_bias);
}

// The shapes, and what a launch of each takes in us: rounds of workgroups times (around + step of 64 * steps [+ gelu]) + launch,
// where a step costs more or less as the CUs fill up.  Fitted to the products of a transformer block (1024 -> 3072, 1024 -> 1024,
// 1024 -> 4096 with GELU, 4096 -> 1024) of 200 - 8500 rows, run in a chain with weights that come from memory; what it picks
// is 0.1 us off the best of all shapes on average.
struct Shape {
    int bm, bn, per_cu;                               // (per_cu: workgroups a CU holds)
    double around, step, step_full, gelu, launch;
};
constexpr Shape kShapes[] = {
    {64, 64, 2, -0.97, 0.502, -0.090, 0.44, 3.73},    // few rows: the most workgroups
    {128, 128, 1, 1.50, 0.448, -0.058, 1.64, 1.45},
    {128, 192, 1, 2.85, 0.576, -0.171, 2.75, 1.50},
    {256, 128, 1, 1.84, 0.743, -0.191, 3.59, 0.73},
    {192, 256, 1, 2.65, 1.244, -0.282, 4.97, 2.68},
    {256, 256, 1, 1.14, 1.543, -0.258, 6.43, 2.61},   // many: the fewest bytes per multiplication
};
// sums of shares: fp32 is written and read where 16-bit results were (us a byte)
constexpr double kSplitBytes = 0.146e-6;

double estimate(const Shape &s, int64_t rows, int64_t K, int64_t N, int act, int splits = 1) {
    const double tiles = static_cast<double>(ceil_div(rows, s.bm) * ceil_div(N, s.bn) * splits), cus = cu_count(), share = tiles / (cus * s.per_cu);
    const double rounds = s.per_cu == 1 ? std::ceil(share) : share < 1 ? (share > 0.5 ? share : 0.5) : share + 0.25;
    const double steps = std::ceil(static_cast<double>(K) / 64 / splits), fill = tiles < cus ? tiles / cus : 1.0;
    const double extra = splits > 1 ? kSplitBytes * static_cast<double>(rows) * static_cast<double>(N) * (8.0 * splits - 4.0) : 0.0;
    return rounds * (s.around + steps * (s.step + s.step_full * fill) + (act ? s.gelu : 0.0)) + s.launch + extra;
}
// Of a launch with GELU in 256 x 256 tiles: the rows that make whole rounds, and the rows of a tile (of 128 columns) in which what is left
// of them is no more than one round.  0: it is more, or nothing.
// A round of few 256 x 256 tiles takes as long as any other.  us, 256 x 256 alone and like this: 1024 -> 4096, 25 536 rows (6.3 rounds) 239.5
// and 227.1, 17 578 (4.3, what is left in 256 x 128) 170.7 and 156.1; 768 -> 3072, 23 437 rows (4.3) 141.7 and 130.0, 28 645 (5.3) 170.1 and
// 159.3.  With more left it gains nothing: 1024 -> 4096, 19 152 rows (4.7) in 128 x 128 175.4 and 177.0.
struct Rounds {
    int64_t whole;
    int rest;
};
Rounds whole_rounds(int64_t rows, int64_t N) {
    const int64_t cols = ceil_div(N, 256), cus = cu_count(), rounds = ceil_div(rows, 256) * cols / cus, whole = rounds * cus / cols * 256;
    if (whole < rows)
        for (const int bm : {128, 256})
            if (ceil_div(rows - whole, bm) * ceil_div(N, 128) <= cus) return {whole, bm};
    return {0, 0};
}

// From here on (outputs) a launch is limited by power, which the estimate knows nothing of: the shape that moves the fewest bytes.
// 25 536 rows, 1024 -> 4096 with GELU: 251 us, 256 x 128 257, 192 x 256 262 (the library and GELU 286; these with 32x32x16).
// With GELU from 4e7 on, where what is left of whole rounds goes in smaller tiles (whole_rounds).  us, the estimate's shape and this: 1024 ->
// 4096, 9887 rows 95.3 and 91.0, 10 375 107.1 and 101.7, 11 962 111.1 and 106.8; 768 -> 3072, 13 834 rows 88.1 and 84.3; 384 -> 1536, 29 817
// rows 88.3 and 59.0.  Below, forwards do not gain (12 frames, 3.9e7: 28.71 and 28.79 ms).
// Up to 7e7 not where tiles of 256 columns compute more than an eighth for nothing (1536 -> 384, 107 523 rows 155 and 203) or the product
// narrows (3072 -> 768, 54 340 rows 276 and 334), nor where 256 x 128 tiles gain more than 15 % by the estimate: a last round of 256 x 256 that is
// half empty and not split (768 -> 3072, 13 342 rows 87 and 98).
constexpr double kTall = 7e7, kTallGelu = 4e7;
constexpr int kLargest = static_cast<int>(sizeof(kShapes) / sizeof(kShapes[0])) - 1, kHalfOfLargest = 3;
static_assert(kShapes[kLargest].bm == 256 && kShapes[kLargest].bn == 256 && kShapes[kHalfOfLargest].bm == 256 && kShapes[kHalfOfLargest].bn == 128);
bool widens(int64_t K, int64_t N) { return K <= N && ceil_div(N, 256) * 256 * 8 <= N * 9; }
int best_shape(int64_t rows, int64_t K, int64_t N, int act) {
    const double outputs = static_cast<double>(rows) * static_cast<double>(N);
    if (outputs >= kTall) return kLargest;
    if (act == COME_ACT_GELU && outputs >= kTallGelu && widens(K, N) &&
        (whole_rounds(rows, N).whole > 0 || estimate(kShapes[kLargest], rows, K, N, act) <= 1.15 * estimate(kShapes[kHalfOfLargest], rows, K, N, act)))
        return kLargest;
    int best = 0;
    for (int i = 1; i <= kLargest; ++i)
        if (estimate(kShapes[i], rows, K, N, act) < estimate(kShapes[best], rows, K, N, act)) best = i;
    return best;
}

template <int DT, int BM, int BN, int QM, int QN, int S, bool SPLIT>
void launch(LinearArgs a, int act, hipStream_t s) {
    a.m_tiles = static_cast<int>(ceil_div(a.rows, BM));
    a.n_tiles = static_cast<int>(ceil_div(a.N, BN));
    a.per_xcd = static_cast<int>(ceil_div(static_cast<int64_t>(a.m_tiles) * a.n_tiles * (SPLIT ? a.splits : 1), 8));
    const dim3 grid(static_cast<unsigned>(8 * a.per_xcd)), block(64 * QM * QN);
    if constexpr (!SPLIT)
        if (act == COME_ACT_GELU) {
            hipLaunchKernelGGL((linear_kernel<DT, BM, BN, QM, QN, S, COME_ACT_GELU, false>), grid, block, 0, s, a);
            return;
        }
    hipLaunchKernelGGL((linear_kernel<DT, BM, BN, QM, QN, S, COME_ACT_NONE, SPLIT>), grid, block, 0, s, a);
}

template <int DT>
void launch_mixed(LinearArgs a, const Rounds &r, hipStream_t s) {
    LinearArgs b = a;
    a.rows = static_cast<int>(r.whole);
    b.rows -= a.rows;
    b.x += r.whole * a.K * 2;
    b.out += r.whole * a.N;
    auto tiles = [](LinearArgs &p, int bm, int bn) {
        p.m_tiles = static_cast<int>(ceil_div(p.rows, bm));
        p.n_tiles = static_cast<int>(ceil_div(p.N, bn));
        p.per_xcd = static_cast<int>(ceil_div(static_cast<int64_t>(p.m_tiles) * p.n_tiles, 8));
    };
    tiles(a, 256, 256);
    tiles(b, r.rest, 128);
    const dim3 grid(static_cast<unsigned>(8 * (a.per_xcd + b.per_xcd)));
    if (r.rest == 128) hipLaunchKernelGGL((linear_mixed_kernel<DT, 128, 128, 2, 4, 4>), grid, dim3(512), 0, s, a, b);
    else hipLaunchKernelGGL((linear_mixed_kernel<DT, 256, 128, 4, 2, 3>), grid, dim3(512), 0, s, a, b);
}

template <int DT>
void launch_shape(int shape, const LinearArgs &a, int act, hipStream_t s) {
    switch (shape) {
        case 0: launch<DT, 64, 64, 2, 2, 4, false>(a, act, s); break;
        case 1: launch<DT, 128, 128, 2, 4, 4, false>(a, act, s); break;
        case 2: launch<DT, 128, 192, 4, 2, 3, false>(a, act, s); break;
        case 3: launch<DT, 256, 128, 4, 2, 3, false>(a, act, s); break;
        case 4: launch<DT, 192, 256, 2, 4, 2, false>(a, act, s); break;
        default: launch<DT, 256, 256, 2, 4, 2, false>(a, act, s); break;
    }
}

// The shapes that shares of K run in.
constexpr int kSplitShapes[] = {0, 1, 3};
template <int DT>
void launch_split(int shape, const LinearArgs &a, hipStream_t s) {
    switch (shape) {
        case 0: launch<DT, 64, 64, 2, 2, 4, true>(a, COME_ACT_NONE, s); break;
        case 1: launch<DT, 128, 128, 2, 4, 4, true>(a, COME_ACT_NONE, s); break;
        default: launch<DT, 256, 128, 4, 2, 3, true>(a, COME_ACT_NONE, s); break;
    }
}

struct SplitPlan {
    int splits, shape;
    double us;
};
SplitPlan split_plan(int64_t rows, int64_t K, int64_t N) {
    SplitPlan best{1, 0, 1e30};
    for (const int splits : {2, 4})
        for (const int i : kSplitShapes) {
            if (K / 64 < 4 * splits) continue;
            const double us = estimate(kShapes[i], rows, K, N, COME_ACT_NONE, splits);
            if (us < best.us) best = SplitPlan{splits, i, us};
        }
    return best;
}

int check_linear(const char *who, const void *x, const void *weight, const void *bias, int dtype, int64_t rows, int64_t in_features,
                 int64_t out_features, const void *out) {
    COME_REQUIRE(dtype == COME_BF16 || dtype == COME_F16, COME_ERR_UNSUPPORTED, "%s: only fp16 and bf16 are supported", who);
    COME_REQUIRE(rows >= 0 && in_features > 0 && out_features > 0, COME_ERR_INVALID, "%s: bad sizes", who);
    COME_REQUIRE(in_features % 64 == 0 && out_features % 8 == 0, COME_ERR_UNSUPPORTED,
                 "%s: in_features must be a multiple of 64 and out_features one of 8", who);
    // byte offsets inside a tile are 32-bit, tiles are counted with 32 bits
    COME_REQUIRE(in_features < (1ll << 22) && rows < (1ll << 31) && out_features < (1ll << 31) &&
                     ceil_div(rows, 64) * ceil_div(out_features, 64) < (1ll << 28),
                 COME_ERR_UNSUPPORTED, "%s: problem too large", who);
    if (rows == 0) return COME_OK;
    COME_REQUIRE(x != nullptr && weight != nullptr && out != nullptr, COME_ERR_INVALID, "%s: NULL tensor", who);
    const void *aligned[] = {x, weight, bias, out};
    for (const void *p : aligned)
        COME_REQUIRE((reinterpret_cast<uintptr_t>(p) & 15) == 0, COME_ERR_INVALID, "%s: pointers must be 16-byte aligned", who);
    return COME_OK;
}

}  // namespace
}  // namespace come

extern "C" int come_linear_is_faster(int64_t rows, int64_t in_features, int64_t out_features, int act) {
    using namespace come;
    if (rows <= 0 || in_features <= 0 || out_features <= 0 || in_features % 64 != 0 || out_features % 8 != 0) return 0;
    const double outputs = static_cast<double>(rows) * static_cast<double>(out_features);
    // us, the library's minus this one's, in a chain of blocks with weights that come from memory.  The library's times jump from
    // one size to the next (1024 -> 4096 with GELU: 31.9 us for 2200 rows, 24.1 for 2400, 31.0 for 3200), so the lines lie where the
    // sizes around them turn, and single sizes inside lose.
    // GELU behind the product as an operation of its own costs a pass over its output.  1024 -> 4096: 6.5 (200 rows), 5.2 (700), 6.1
    // (1596), 6.3 (2200), -2 (2400), 1.8 (3200), 9.0 (4300), 5.6 (5000), -3 (6200 - 6600), 8.6 (7000), 9.6 (8000), 40 (9600); 768 ->
    // 3072: 6.2 (1596), 18 (6400), -6 and 1 (8500), 10 (10 240); 384 -> 1536: 10 (10 240), 15 (17 000), -6 (19 152), 20 (21 000).
    // Beyond, forwards are limited by power.  ms, the library and this: 10 374 rows 33.10 and 32.65, 11 172 36.99 and 35.99, 11 970 39.67 and
    // 38.49; 12 768 42.93 and 42.50, 14 364 48.88 and 48.37, 15 960 54.78 and 54.20, which is 1 % and about what the runs differ by: 5e7 - 7e7
    // stay with the library.
    // Not for K above 1024 between 4e7 and 5e7, where the library is as good: us, the library and this, 1536 -> 6144, 6591 rows 144 and 129, 6998
    // 148 and 153, 7486 155 and 155; 2048 -> 8192, 4943 195 and 163, 5249 179 and 190, 6042 193 and 203.
    // From 7e7 on longer K gains as well: 1536 -> 6144, 11 635 rows 248 and 213, 17 225 380 and 321, 32 683 623 and 599; 2048 -> 8192, 8746 rows 276 and
    // 285, 12 953 458 and 402, 24 545 733 and 743; 4096 -> 4096, 17 413 rows 571 and 485, 34 197 1025 and 1035 (48 959 1232 and 1454).
    // Not for products that narrow, from 4e7 on: 4096 -> 1024, 41 992 rows 303 and 399, 74 218 505 and 661, 102 539 784 and 867.
    if (act == COME_ACT_GELU) return outputs <= 4e7 || (widens(in_features, out_features) && ((outputs <= 5e7 && in_features <= 1024) || outputs >= kTall));
    // 1024 -> 3072: 4.4 (200 rows), 2.6 (1596), 2.5 and 3.6 (2400), -1.6 and -1.0 (2600), -3.0 (2800), -2 (3200 - 4600), -3.9 (5000);
    // 768 -> 2304: 4.8 and 5.2 (2800), -0.9 (3600); 384 -> 1152: 8.9 (6400); 1024 -> 1024: 3.0 (200), 3.0 (1596), 2.5 (3600), 1.8 (6400),
    // 2.5 (7000), -0.5 (7300), -1.2 and 1.5 (7500), -6.4 (8500).
    if (in_features <= 2048) return outputs <= 7.4e6;
    // With the residual step behind, in shares where that is better.  4096 -> 1024: 2.0 (200), 5.7 (700), 5.7 (1596), 3.6 (2000), 1.1 (2200),
    // 0.6 and 0.1 (2400), -3.3 (2800), -3.1 (3000), 3.0 (3100), 3.9 (3200), 1.4 (3600), 2.4 (4000), 3.5 (4300), 0.5 (5000), 1.7 (5100),
    // -4.9 (5500), -24 (8500); 3072 -> 768: 0.7 (1596), 2.8 (2200), 2.4 (2600), -0.9 (2800), -3.0 (3600), 1.1 (4200), -0.9 (5000, 6400).
    // Forwards of 3 frames, this one's and the library's: 8.82 and 8.95 ms (2394 rows), 9.75 and 9.69 (2800).
    if (in_features < 4096) return outputs <= 2.1e6;
    return outputs <= 2.5e6 || (outputs >= 3.1e6 && outputs <= 5.3e6);
}

// Shares of K for a product whose sums come_residual_norm_split takes (1: no shares).
extern "C" int come_linear_splits(int64_t rows, int64_t in_features, int64_t out_features) {
    using namespace come;
    if (rows <= 0 || in_features <= 0 || out_features <= 0 || in_features % 64 != 0 || out_features % 8 != 0) return 1;
    const SplitPlan p = split_plan(rows, in_features, out_features);
    const double whole = estimate(kShapes[best_shape(rows, in_features, out_features, COME_ACT_NONE)], rows, in_features, out_features, COME_ACT_NONE);
    return p.us < whole && come_linear_is_faster(rows, in_features, out_features, COME_ACT_NONE) ? p.splits : 1;
}

extern "C" int come_linear(const void *x, const void *weight, const void *bias, int dtype, int64_t rows, int64_t in_features,
                           int64_t out_features, int act, void *out, void *stream) {
    using namespace come;
    clear_error();
    COME_REQUIRE(act == COME_ACT_NONE || act == COME_ACT_GELU, COME_ERR_INVALID, "come_linear: unknown activation %d", act);
    if (const int status = check_linear("come_linear", x, weight, bias, dtype, rows, in_features, out_features, out)) return status;
    if (rows == 0) return COME_OK;
    LinearArgs a{};
    a.x = static_cast<const char *>(x);
    a.w = static_cast<const char *>(weight);
    a.bias = static_cast<const uint16_t *>(bias);
    a.out = static_cast<uint16_t *>(out);
    a.rows = static_cast<int>(rows);
    a.K = static_cast<int>(in_features);
    a.N = static_cast<int>(out_features);
    const int shape = best_shape(rows, in_features, out_features, act);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Rounds rounds = act == COME_ACT_GELU && shape == kLargest ? whole_rounds(rows, out_features) : Rounds{};
    if (rounds.whole > 0 && dtype == COME_BF16) launch_mixed<COME_BF16>(a, rounds, s);
    else if (rounds.whole > 0) launch_mixed<COME_F16>(a, rounds, s);
    else if (dtype == COME_BF16) launch_shape<COME_BF16>(shape, a, act, s);
    else launch_shape<COME_F16>(shape, a, act, s);
    COME_CHECK_LAUNCH("come_linear");
    return COME_OK;
}

extern "C" int come_linear_split(const void *x, const void *weight, int dtype, int64_t rows, int64_t in_features, int64_t out_features,
                                 int splits, float *partial, void *stream) {
    using namespace come;
    clear_error();
    if (const int status = check_linear("come_linear_split", x, weight, nullptr, dtype, rows, in_features, out_features, partial)) return status;
    COME_REQUIRE((splits == 2 || splits == 4) && in_features / 64 >= 4 * splits, COME_ERR_INVALID,
                 "come_linear_split: 2 or 4 shares of at least 256 features each");
    if (rows == 0) return COME_OK;
    LinearArgs a{};
    a.x = static_cast<const char *>(x);
    a.w = static_cast<const char *>(weight);
    a.partial = partial;
    a.rows = static_cast<int>(rows);
    a.K = static_cast<int>(in_features);
    a.N = static_cast<int>(out_features);
    a.splits = splits;
    int shape = kSplitShapes[0];
    for (const int i : kSplitShapes)
        if (estimate(kShapes[i], rows, in_features, out_features, COME_ACT_NONE, splits) <
            estimate(kShapes[shape], rows, in_features, out_features, COME_ACT_NONE, splits))
            shape = i;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == COME_BF16) launch_split<COME_BF16>(shape, a, s);
    else launch_split<COME_F16>(shape, a, s);
    COME_CHECK_LAUNCH("come_linear_split");
    return COME_OK;
}
