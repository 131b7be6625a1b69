// Window confidence means, lowest-confidence window selection and the merge plan for gfx950.
//
// One workgroup per batch element: it reduces every full window of that element's frames to its mean, finds the
// lower of the two order statistics that torch.quantile's linear interpolation needs with an exact radix select,
// its upper neighbour with one more reduction, forms the threshold in fp32, writes the strict "mean < threshold"
// mask and - when asked to - turns the mask into the packed-row plan of the merge (per-window prefix, row lengths,
// row offsets) without leaving the kernel.
//
// The data is tiny (thousands of means) and lives on one CU, so the kernel is priced in issued instructions and dependent
// steps, not in bytes.  Hence: a thread keeps the ordered keys of its windows in registers, cross-lane reductions and scans are
// DPP moves instead of LDS permutes, a radix pass is "count, barrier, one wavefront scans the 1024-bin histogram, barrier", the
// bins of the first digit divide the range between the least and the largest key, and a bin of few keys is ranked by
// comparison; with a plan, comparison and plan share one sweep in which a wavefront's ballot over 64 windows of a row gives
// their packed positions.  Up to kFewWindows windows take a kernel of their own, the means of more than kManyWindows a launch in
// front.  Selection alone from smooth fp32 confidences, us: 80 windows 2.9, 576 4.1, 2304 5.8, 4608 7.9, 13 824 14.0, 28 800 19.2.
#include "come_common.h"

#include <cmath>

namespace come {
namespace {

constexpr int kSelectThreads = 1024;
constexpr int kSelectWaves = kSelectThreads / 64;
constexpr int kLdsKeys = 16384;             // windows per batch element whose keys fit in LDS (global memory beyond)
constexpr int kBinBits = 10;
constexpr int kBins = 1 << kBinBits;
constexpr int kBinsPerLane = kBins / 64;
constexpr int kMaxPasses = 4;               // 32 key bits in digits of 10
constexpr int kCandidates = 64;             // a bin of at most this many keys is not split any further: a lane per key

__device__ inline uint32_t ordered_key(float x) {           // monotone float -> uint32
    const uint32_t u = __float_as_uint(x);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline float key_to_float(uint32_t k) {
    const uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
    return __uint_as_float(u);
}

#define COME_WAVE_REDUCE(NAME, EXPR)                                                   \
    __device__ inline uint32_t NAME(uint32_t v) {                                      \
        uint32_t t;                                                                    \
        t = dpp_take<kRowShr1, 0xf>(v, v); v = EXPR;                                   \
        t = dpp_take<kRowShr2, 0xf>(v, v); v = EXPR;                                   \
        t = dpp_take<kRowShr4, 0xf>(v, v); v = EXPR;                                   \
        t = dpp_take<kRowShr8, 0xf>(v, v); v = EXPR;                                   \
        t = dpp_take<kRowBcast15, 0xa>(v, v); v = EXPR;                                \
        t = dpp_take<kRowBcast31, 0xc>(v, v); v = EXPR;                                \
        return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63)); \
    }
COME_WAVE_REDUCE(wave_min, min(v, t))
COME_WAVE_REDUCE(wave_max, max(v, t))
#undef COME_WAVE_REDUCE
__device__ inline uint32_t wave_sum(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(wave_scan_add(v)), 63));
}

struct alignas(16) SelectShared {
    uint32_t hist[kMaxPasses][kBins];       // one histogram per pass, all cleared up front
    uint32_t keys[kLdsKeys];                // ordered keys of the window means
    uint32_t red[2][kSelectWaves];          // per wavefront: least and largest key
    uint32_t found[3];                      // per pass: bin that holds rank k, keys in front of it, keys in it
    uint32_t above;                         // smallest key above the lower order statistic, or above the candidates
    uint32_t n_cand, cand[kCandidates];     // keys of a bin that holds few
    float fred[kSelectWaves + 1];
};

// Workgroup-wide sum (every thread receives it).
__device__ float block_sum(float v, float *red) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < kSelectWaves; ++w) t += red[w];
    return t;
}

template <int DT> __device__ inline float round_dt(float x) {
    if (DT == COME_BF16) return __uint_as_float(pack2_bf16(x, 0.f) << 16);
    return x;
}

// torch.lerp of the two order statistics
__device__ inline float lerp_as_torch(float va, float vb, float frac) {
    const float diff = __fsub_rn(vb, va);
    return frac < 0.5f ? __fadd_rn(va, __fmul_rn(frac, diff)) : __fsub_rn(vb, __fmul_rn(diff, __fsub_rn(1.0f, frac)));
}

struct SelectArgs {
    const void *conf;
    int frames, H, W, gh, gw;
    int mode;
    float threshold;
    int rank_lo, rank_hi;
    float frac;
    float *means;
    uint8_t *mask;
    // merge plan (offsets == nullptr: selection only)
    int32_t *offsets, *prefix;
    int start, tail;
    int given;                              // the means have been computed (window_means_kernel)
    uint64_t *post;                         // host memory that receives the packed row count (nullptr: not posted)
    uint32_t post_tag;
    FastDiv by_windows, by_mw;              // windows per frame, windows per grid row
};

// k-th smallest (0-based) ordered key of the keys of this workgroup; visit(f) calls f(key) for every key the
// calling thread owns.  All threads call it and all receive the key.  One barrier for the bits in which the keys
// differ, then two per pass: the keys are counted into the pass's histogram, wavefront 0 scans it and publishes the
// bin that holds rank k.  Distinct fp32 means leave a handful of keys in that bin after the first pass: those are
// collected (one barrier) and ranked by comparison, which also gives the key of rank k + 1 (`has_next`; the smallest key
// above the bin where it holds no further one) instead of two more passes and one over all keys for the neighbour.
// DROP: low key bits that only repeat the sign (16 for bf16 means).
template <bool COLLECT, int DROP, typename Visit>
__device__ uint32_t select_kth(SelectShared &sh, Visit visit, uint32_t k, uint32_t &next, bool &has_next) {
    has_next = false;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    constexpr int drop = DROP;
    uint32_t least = 0xffffffffu, most = 0u;
    visit([&](uint32_t key) {
        least = min(least, key);
        most = max(most, key);
    });
    least = wave_min(least);
    most = wave_max(most);
    if (lane == 0) {
        sh.red[0][wave] = least;
        sh.red[1][wave] = most;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kSelectWaves; ++w) {
        least = min(least, sh.red[0][w]);
        most = max(most, sh.red[1][w]);
    }
    // The bins of the first digit divide the range that the keys are spread over.  (Bins by key bits alone leave five of 1024 to
    // keys between 1 and 2.5, which differ in their highest exponent bit: an addition to LDS at one address costs 35 cycles, one
    // after another.  Selection, us: 576 windows 5.1 -> 4.5, 2304 7.3 -> 6.0, 13 824 22.8 -> 19.7.)
    uint32_t lo = least >> drop;                                                    // (shifted keys)
    const uint32_t range = (most >> drop) - lo;
    int width = range == 0 ? 0 : 32 - __clz(static_cast<int>(range));               // candidates: lo .. lo + 2^width - 1
    int shift = width > kBinBits ? width - kBinBits : 0;
#pragma unroll 1
    for (int pass = 0; pass < kMaxPasses; ++pass) {
        const uint32_t limit = width >= 32 ? 0xffffffffu : (1u << width) - 1u;
        uint32_t *hist = sh.hist[pass];
        visit([&](uint32_t key) {
            const uint32_t rel = (key >> drop) - lo;
            if (rel <= limit) atomicAdd(&hist[rel >> shift], 1u);
        });
        __syncthreads();
        if (wave == 0) {            // lane l owns bins kBinsPerLane * l .. + kBinsPerLane - 1
            uint32_t c[kBinsPerLane];
            uint32_t s = 0;
#pragma unroll
            for (int j = 0; j < kBinsPerLane; j += 4) {
                const uint4 q = *reinterpret_cast<const uint4 *>(&hist[lane * kBinsPerLane + j]);
                c[j] = q.x;
                c[j + 1] = q.y;
                c[j + 2] = q.z;
                c[j + 3] = q.w;
                s += q.x + q.y + q.z + q.w;
            }
            const uint32_t incl = wave_scan_add(s);
            const uint32_t excl = incl - s;
            if (k >= excl && k < incl) {        // exactly one lane: its bin that holds rank k, the keys in front of it
                uint32_t bin = static_cast<uint32_t>(lane * kBinsPerLane), before = excl;
                uint32_t run = excl, behind = incl;             // keys up to the end of the bin
#pragma unroll
                for (int j = 0; j < kBinsPerLane - 1; ++j) {
                    run += c[j];
                    const bool past = k >= run;
                    bin += past ? 1u : 0u;
                    before = past ? run : before;
                    behind = past ? behind : min(behind, run);
                }
                sh.found[0] = bin;
                sh.found[1] = before;
                if (COLLECT) sh.found[2] = behind - before;
            }
        }
        __syncthreads();
        k -= sh.found[1];
        lo += sh.found[0] << shift;
        if (shift == 0) break;
        const uint32_t count = COLLECT ? static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(sh.found[2]))) : 0;
        if (COLLECT && count <= kCandidates) {
            const uint32_t span = 1u << shift;
            uint32_t above = 0xffffffffu;
            visit([&](uint32_t key) {
                const uint32_t at = key >> drop;
                if (at >= lo) {
                    if (at - lo < span) sh.cand[atomicAdd(&sh.n_cand, 1u)] = key;
                    else above = min(above, key);
                }
            });
            above = wave_min(above);
            if (lane == 0) atomicMin(&sh.above, above);
            __syncthreads();
            const uint32_t mine = static_cast<uint32_t>(lane) < count ? sh.cand[lane] : 0xffffffffu;
            uint32_t rank = 0;                              // by key, then by place
            for (uint32_t j = 0; j < count; ++j) {
                const uint32_t other = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(mine), static_cast<int>(j)));
                rank += (other < mine || (other == mine && j < static_cast<uint32_t>(lane))) ? 1u : 0u;
            }
            auto of_rank = [&](uint32_t r) {                // (exactly one of the lanes below `count` has it)
                const int l = __builtin_ctzll(__ballot(static_cast<uint32_t>(lane) < count && rank == r));
                return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(mine), l));
            };
            has_next = true;
            next = k + 1 < count ? of_rank(k + 1) : sh.above;
            return of_rank(k);
        }
        width = shift;
        shift = shift > kBinBits ? shift - kBinBits : 0;
    }
    return DROP == 0 || (lo >> (31 - DROP)) != 0 ? lo << drop : (lo << drop) | ((1u << drop) - 1u);       // (negative numbers have their bits inverted)
}

// Mean of window i of a batch element (modes 0 and 1), as step 1 of select_windows_kernel forms it.
template <int DT, int GH, int GW>
__device__ inline float window_mean(const SelectArgs &a, int64_t conf_first, int i, int M, int mw) {
    using V = Vec16<DT>;
    const int gh = GH > 0 ? GH : a.gh, gw = GW > 0 ? GW : a.gw;
    const int f = static_cast<int>(fast_div(i, a.by_windows)), m = i - f * M;
    const int wy = static_cast<int>(fast_div(m, a.by_mw)), wx = m - wy * mw;
    const int64_t base = conf_first + static_cast<int64_t>(f) * a.H * a.W + (wy * gh) * a.W + wx * gw;
    float acc = 0.f;
    if constexpr (GH > 0) {
        float x[GH * GW];
#pragma unroll
        for (int dy = 0; dy < GH; ++dy)
#pragma unroll
            for (int dx = 0; dx < GW; ++dx) x[dy * GW + dx] = V::load1(a.conf, base + dy * a.W + dx);
#pragma unroll
        for (int t = 0; t < GH * GW; ++t) acc = __fadd_rn(acc, x[t]);
    } else {
        for (int dy = 0; dy < gh; ++dy)
            for (int dx = 0; dx < gw; ++dx) acc = __fadd_rn(acc, V::load1(a.conf, base + dy * a.W + dx));
    }
    return round_dt<DT>(__fdiv_rn(acc, static_cast<float>(gh * gw)));
}

// The means of many windows, a thread each over the whole chip (modes 0 and 1): nine strided loads a window are 15 000 cycles of
// one CU's address unit for 13 824 windows.  Selection, us: 13 824 windows 17.0 -> 14.0, 9216 12.0 -> 10.8, 4608 9.0 -> 9.3 (and 7.9
// without it, with eight keys a thread).
constexpr int kManyWindows = 8 * kSelectThreads;
template <int DT, int GH, int GW>
__global__ __launch_bounds__(256) void window_means_kernel(const SelectArgs a) {
    const int mw = a.W / (GW > 0 ? GW : a.gw), M = a.H / (GH > 0 ? GH : a.gh) * mw, n = a.frames * M;
    const int i = static_cast<int>(blockIdx.x * 256 + threadIdx.x);
    if (i >= n) return;
    const int64_t batch = blockIdx.y;
    a.means[batch * n + i] = window_mean<DT, GH, GW>(a, batch * a.frames * a.H * a.W, i, M, mw);
}

// Few windows by rank (mode 0, no plan): a key per thread, whose rank is the number of smaller keys; the lower order statistic is
// the largest key with a rank of at most rank_lo, the upper one that of rank_hi.  Three barriers instead of eight, no histogram.
// With the histogram, us: 25 windows 4.8 -> 2.4, 80 5.4 -> 2.9, 144 5.4 -> 3.7; from about 190 on the kernel below is as fast.
constexpr int kFewWindows = 192;
template <int DT, int GH, int GW>
__global__ __launch_bounds__(kFewWindows) void select_few_kernel(const SelectArgs a) {
    __shared__ __attribute__((aligned(16))) uint32_t keys[kFewWindows];
    __shared__ uint32_t found[2];
    const int mw = a.W / (GW > 0 ? GW : a.gw), M = a.H / (GH > 0 ? GH : a.gh) * mw, n = a.frames * M;
    const int64_t batch = blockIdx.x;
    const int i = static_cast<int>(threadIdx.x);
    const float mean = window_mean<DT, GH, GW>(a, batch * a.frames * a.H * a.W, min(i, n - 1), M, mw);
    const uint32_t mine = ordered_key(mean);
    keys[i] = i < n ? mine : 0xffffffffu;                   // (counts as smaller than nothing)
    if (i < 2) found[i] = 0;
    if (a.means != nullptr && i < n) a.means[batch * n + i] = mean;
    __syncthreads();
    int less = 0;
    for (int j = 0; j < n; j += 32) {                       // (the launch has whole wavefronts: keys up to a multiple of 64)
        uint4 k[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) k[u] = *reinterpret_cast<const uint4 *>(&keys[j + 4 * u]);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            less += (k[u].x < mine ? 1 : 0) + (k[u].y < mine ? 1 : 0) + (k[u].z < mine ? 1 : 0) + (k[u].w < mine ? 1 : 0);
    }
    const uint32_t lo = wave_max(i < n && less <= a.rank_lo ? mine : 0u), hi = wave_max(i < n && less <= a.rank_hi ? mine : 0u);
    if ((i & 63) == 0) {
        atomicMax(&found[0], lo);
        atomicMax(&found[1], hi);
    }
    __syncthreads();
    if (i < n) {
        const float va = key_to_float(found[0]), vb = key_to_float(found[1]);
        a.mask[batch * n + i] = mean < lerp_as_torch(va, vb, a.frac) ? 1 : 0;
    }
}

// KEYS: windows per thread whose keys stay in its registers (at most KEYS * 1024 windows), 0: any number, through global memory.
// A sweep over keys in LDS, one after another, took a wavefront 440 cycles a key (13 824 windows: 6 - 12 thousand cycles each of
// four sweeps), and the loads of a window's values waited for those of the one before.  Selection, us, keys in LDS -> in
// registers: 576 windows 4.5 -> 4.1, 2880 7.1 -> 6.3, 13 824 19.7 -> 17.0; 18 432 (keys in global memory) 26.4 -> 16.0.
template <int DT, int GH, int GW, int KEYS>
__global__ __launch_bounds__(kSelectThreads) void select_windows_kernel(const SelectArgs a) {
    constexpr bool COLLECT = DT == COME_F32;
    using V = Vec16<DT>;
    __shared__ SelectShared sh;

    const int H = a.H, W = a.W, frames = a.frames, mode = a.mode;
    const int gh = GH > 0 ? GH : a.gh, gw = GW > 0 ? GW : a.gw;
    const int mh = H / gh, mw = W / gw;
    const int M = mh * mw;
    const int n = frames * M;
    const int64_t batch_first = static_cast<int64_t>(blockIdx.x) * n;
    float *my_means = a.means != nullptr ? a.means + batch_first : nullptr;      // (nullptr only while the keys fit in LDS)
    uint8_t *my_mask = a.mask + batch_first;
    constexpr bool in_lds = KEYS > 0 && KEYS * kSelectThreads <= kLdsKeys;           // (of a plan)
    const bool plan = a.offsets != nullptr;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int64_t conf_first = static_cast<int64_t>(blockIdx.x) * frames * H * W;

    for (int i = threadIdx.x; i < kMaxPasses * kBins; i += kSelectThreads) (&sh.hist[0][0])[i] = 0;
    if (threadIdx.x == 0) {
        sh.above = 0xffffffffu;
        sh.n_cand = 0;
    }

    // 0. normalised-score mode: z = (x - mean) / (std + 1e-3) over all positions of the batch element,
    //    every tensor operation of that chain rounded to the confidence dtype (unbiased std)
    float z_mean = 0.f, z_denom = 1.f;
    if (mode == 2) {
        const int64_t T = static_cast<int64_t>(frames) * H * W;
        float acc = 0.f;
        for (int64_t i = threadIdx.x; i < T; i += kSelectThreads) acc += V::load1(a.conf, conf_first + i);
        const float mean32 = block_sum(acc, sh.fred) / static_cast<float>(T);
        acc = 0.f;
        for (int64_t i = threadIdx.x; i < T; i += kSelectThreads) {
            const float d = V::load1(a.conf, conf_first + i) - mean32;
            acc += d * d;
        }
        const float var = block_sum(acc, sh.fred) / static_cast<float>(T > 1 ? T - 1 : 1);
        z_mean = round_dt<DT>(mean32);
        z_denom = round_dt<DT>(round_dt<DT>(sqrtf(var)) + 1e-3f);
    }

    // 1. window means: fp32 running sum in window row-major order, one division, rounded to the confidence dtype
    //    and widened back to fp32.  With a compile-time window shape all loads of several windows are issued before the
    //    first addition waits for one.
    constexpr int kAtOnce = KEYS == 0 || GH == 0 ? 1 : KEYS < 4 ? KEYS : 4;
    constexpr int NW = GH > 0 ? GH * GW : 1;
    uint32_t own[KEYS > 0 ? KEYS : 1];                       // keys of windows threadIdx.x + 1024 u
    auto means_from = [&](int i0, uint32_t *keys) __attribute__((always_inline)) {
        float x[kAtOnce][NW];
        int64_t base[kAtOnce];
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            if (u > 0 && i0 - static_cast<int>(threadIdx.x) + u * kSelectThreads >= n) continue;      // (uniform)
            const int i = min(i0 + u * kSelectThreads, n - 1);       // (a window beyond the end is computed twice, stored once)
            const int f = static_cast<int>(fast_div(i, a.by_windows));
            const int m = i - f * M;
            const int wy = static_cast<int>(fast_div(m, a.by_mw));
            const int wx = m - wy * mw;
            base[u] = conf_first + static_cast<int64_t>(f) * H * W + (wy * gh) * W + wx * gw;
            if constexpr (GH > 0) {
#pragma unroll
                for (int dy = 0; dy < GH; ++dy)
#pragma unroll
                    for (int dx = 0; dx < GW; ++dx) x[u][dy * GW + dx] = V::load1(a.conf, base[u] + dy * W + dx);
            }
        }
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            if (u > 0 && i0 - static_cast<int>(threadIdx.x) + u * kSelectThreads >= n) continue;
            const int i = i0 + u * kSelectThreads;
            float acc = 0.f;
            if constexpr (GH > 0) {
#pragma unroll
                for (int t = 0; t < GH * GW; ++t) {
                    float v = x[u][t];
                    if (mode == 2) v = round_dt<DT>(__fdiv_rn(round_dt<DT>(__fsub_rn(v, z_mean)), z_denom));
                    acc = __fadd_rn(acc, v);
                }
            } else {
                for (int dy = 0; dy < gh; ++dy)
                    for (int dx = 0; dx < gw; ++dx) {
                        float v = V::load1(a.conf, base[u] + dy * W + dx);
                        if (mode == 2) v = round_dt<DT>(__fdiv_rn(round_dt<DT>(__fsub_rn(v, z_mean)), z_denom));
                        acc = __fadd_rn(acc, v);
                    }
            }
            const float mean = round_dt<DT>(__fdiv_rn(acc, static_cast<float>(gh * gw)));
            if (KEYS > 0) keys[u] = ordered_key(mean);
            if (i < n) {
                if (my_means != nullptr) my_means[i] = mean;
                if (in_lds && plan) sh.keys[i] = keys[u];
            }
        }
    };
    if (KEYS > 8 && a.given) {
#pragma unroll
        for (int u = 0; u < KEYS; ++u) {
            const int i = static_cast<int>(threadIdx.x) + u * kSelectThreads;
            if (u * kSelectThreads < n && i < n) own[u] = __float_as_uint(my_means[i]);
        }
#pragma unroll
        for (int u = 0; u < KEYS; ++u) {
            const int i = static_cast<int>(threadIdx.x) + u * kSelectThreads;
            if (u * kSelectThreads < n) {
                own[u] = ordered_key(__uint_as_float(own[u]));
                if (in_lds && plan && i < n) sh.keys[i] = own[u];
            }
        }
    } else if constexpr (KEYS > 0) {
#pragma unroll
        for (int u0 = 0; u0 < KEYS; u0 += kAtOnce)
            if (u0 * kSelectThreads < n) means_from(static_cast<int>(threadIdx.x) + u0 * kSelectThreads, own + u0);
    } else {
        for (int i0 = threadIdx.x; i0 < n && !a.given; i0 += kSelectThreads) means_from(i0, nullptr);
        __syncthreads();                       // the means in global memory are read back by other threads
    }
    auto visit_keys = [&](auto f) __attribute__((always_inline)) {
        if constexpr (KEYS > 0) {
#pragma unroll
            for (int u = 0; u < KEYS; ++u)
                if (u * kSelectThreads < n && static_cast<int>(threadIdx.x) + u * kSelectThreads < n) f(own[u]);
        } else {
            for (int i = threadIdx.x; i < n; i += kSelectThreads) f(ordered_key(my_means[i]));
        }
    };

    // 2. threshold.  Ranking: the two neighbouring order statistics of torch.quantile's linear interpolation;
    //    the upper one is either the same value again (duplicates) or the smallest value above the lower one.
    //    Absolute and normalised score compare a tensor of the confidence dtype with a scalar: the scalar is
    //    rounded to that dtype first, as the tensor library does (a bf16 mean of 0.44921875 is not below 0.45).
    float cut = round_dt<DT>(a.threshold);
    if (mode == 0) {
        uint32_t key_b = 0;
        bool has_b = false;
        const uint32_t key_a = select_kth<COLLECT, DT == COME_BF16 ? 16 : 0>(sh, visit_keys, static_cast<uint32_t>(a.rank_lo), key_b, has_b);
        const float va = key_to_float(key_a);
        float vb = va;
        if (a.rank_hi != a.rank_lo && has_b) {
            vb = key_to_float(key_b);
        } else if (a.rank_hi != a.rank_lo) {
            // counts are integers: exact whatever the number of windows
            uint32_t le = 0;
            uint32_t above = 0xffffffffu;
            visit_keys([&](uint32_t key) {
                if (key <= key_a) ++le;
                else above = min(above, key);
            });
            le = wave_sum(le);
            above = wave_min(above);
            if (lane == 0) {
                sh.red[0][wave] = le;          // free again: its readers passed at least two barriers since
                atomicMin(&sh.above, above);
            }
            __syncthreads();
            uint32_t count_le = 0;
#pragma unroll
            for (int w = 0; w < kSelectWaves; ++w) count_le += sh.red[0][w];
            if (count_le <= static_cast<uint32_t>(a.rank_hi)) vb = key_to_float(sh.above);
        }
        cut = lerp_as_torch(va, vb, a.frac);
    }

    // 3. strict comparison (on the float values: -0 and +0 differ as keys, not as numbers)
    if (!plan) {
        if constexpr (KEYS > 0) {
#pragma unroll
            for (int u = 0; u < KEYS; ++u) {
                const int i = static_cast<int>(threadIdx.x) + u * kSelectThreads;
                if (u * kSelectThreads < n && i < n) my_mask[i] = key_to_float(own[u]) < cut ? 1 : 0;
            }
        } else {
            for (int i = threadIdx.x; i < n; i += kSelectThreads) my_mask[i] = my_means[i] < cut ? 1 : 0;
        }
        return;
    }

    // 3 + 4. with a merge plan: a wavefront takes whole rows (frames), 64 windows at a time, so the comparison
    //    bits of a step are one ballot and give the packed position of every window inside its row
    //    (start_index + G * kept before + merged before) and the row length; with a single batch element the row
    //    offsets follow (otherwise a second small kernel scans the lengths)
    __syncthreads();                                        // keys written by other threads (no barrier yet in modes 1, 2)
    const int G = gh * gw;
    const int row_first = blockIdx.x * frames;
    const uint64_t below = (1ull << lane) - 1ull;
    for (int f = wave; f < frames; f += kSelectWaves) {
        int running = 0;                                    // wave-uniform
        for (int m0 = 0; m0 < M; m0 += 64) {
            const int m = m0 + lane;
            const bool valid = m < M;
            const int i = f * M + min(m, M - 1);
            const float mean = in_lds ? key_to_float(sh.keys[i]) : my_means[i];
            const bool merged = valid && mean < cut;
            if (valid) my_mask[i] = merged ? 1 : 0;
            const uint64_t merged_bits = __ballot(merged);
            const int merged_before = __popcll(merged_bits & below);
            if (valid)
                a.prefix[static_cast<int64_t>(row_first + f) * M + m] =
                    running + merged_before + (lane - merged_before) * G;
            const int n_valid = min(64, M - m0);
            const int n_merged = __popcll(merged_bits);
            running += n_merged + (n_valid - n_merged) * G;
        }
        if (lane == 0) a.offsets[row_first + f + 1] = a.start + a.tail + running;
    }
    if (gridDim.x != 1) return;
    if (threadIdx.x == 0) a.offsets[0] = 0;
    __syncthreads();
    if (wave == 0) {                                        // in-place inclusive scan of the row lengths
        int carry = 0;
        for (int r0 = 0; r0 < frames; r0 += 64) {
            const int r = r0 + lane;
            const uint32_t len = r < frames ? static_cast<uint32_t>(a.offsets[r + 1]) : 0u;
            const uint32_t v = wave_scan_add(len);
            if (r < frames) a.offsets[r + 1] = static_cast<int>(v) + carry;
            carry += __builtin_amdgcn_readlane(static_cast<int>(v), 63);
        }
        if (a.post != nullptr && lane == 0) post_to_host(a.post, a.post_tag, static_cast<uint32_t>(carry));
    }
}

// offsets[0] = 0 and an in-place inclusive scan of the row lengths in offsets[1 .. rows] (one wavefront)
__global__ __launch_bounds__(64) void scan_offsets_kernel(int32_t *__restrict__ offsets, int rows, uint64_t *post,
                                                          uint32_t post_tag) {
    const int lane = threadIdx.x;
    if (lane == 0) offsets[0] = 0;
    int carry = 0;
    for (int r0 = 0; r0 < rows; r0 += 64) {
        const int r = r0 + lane;
        const uint32_t len = r < rows ? static_cast<uint32_t>(offsets[r + 1]) : 0u;
        const uint32_t v = wave_scan_add(len);
        if (r < rows) offsets[r + 1] = static_cast<int>(v) + carry;
        carry += __builtin_amdgcn_readlane(static_cast<int>(v), 63);
    }
    if (post != nullptr && lane == 0) post_to_host(post, post_tag, static_cast<uint32_t>(carry));
}

int select_impl(const char *who, const void *conf, int dtype, int64_t batch, int64_t frames, int64_t grid_h,
                int64_t grid_w, int64_t group_h, int64_t group_w, int mode, float threshold, float *means_f32,
                uint8_t *merge_mask, void *work, int64_t work_bytes, bool plan, int64_t start_index,
                int32_t *offsets, int32_t *group_prefix, void *stream, bool means_optional = false,
                uint64_t *post = nullptr, uint32_t post_tag = 0) {
    COME_REQUIRE(dtype == COME_BF16 || dtype == COME_F32, COME_ERR_UNSUPPORTED, "%s: confidence must be bf16 or fp32",
                 who);
    COME_REQUIRE(batch >= 0 && frames >= 0 && grid_h >= 0 && grid_w >= 0, COME_ERR_INVALID, "%s: negative size", who);
    COME_REQUIRE(group_h > 0 && group_w > 0, COME_ERR_INVALID, "%s: group_h and group_w must be > 0", who);
    COME_REQUIRE(mode >= 0 && mode <= 2, COME_ERR_UNSUPPORTED, "%s: unknown mode %d", who, mode);
    if (mode == 0)
        COME_REQUIRE(threshold >= 0.f && threshold <= 1.f, COME_ERR_INVALID,
                     "%s: ranking mode requires threshold in [0, 1], got %g", who, (double)threshold);
    const int64_t windows = (grid_h / group_h) * (grid_w / group_w);
    const int64_t n = frames * windows;
    const int64_t rows = batch * frames;
    if (plan) {
        COME_REQUIRE(start_index >= 0, COME_ERR_INVALID, "%s: start_index must be >= 0", who);
        COME_REQUIRE(batch > 0 && n > 0, COME_ERR_UNSUPPORTED,
                     "%s: no full window to select from (plan such rows with come_merge_plan)", who);
        COME_REQUIRE(offsets != nullptr && group_prefix != nullptr, COME_ERR_INVALID,
                     "%s: offsets / group_prefix is NULL", who);
        COME_REQUIRE(rows < (1ll << 31) && rows * (start_index + grid_h * grid_w) < (1ll << 31), COME_ERR_UNSUPPORTED,
                     "%s: rows * tokens per row must stay below 2^31", who);
    }
    if (batch == 0 || n == 0) return COME_OK;
    // n < 2^24: the rank float(threshold) * (n - 1) is formed in fp32, as torch.quantile forms it
    COME_REQUIRE(n < (1ll << 24) && batch < (1ll << 31) && frames * grid_h * grid_w < (1ll << 31) &&
                     batch * frames * grid_h * grid_w < (1ll << 40),
                 COME_ERR_UNSUPPORTED, "%s: problem too large", who);
    COME_REQUIRE(conf && merge_mask, COME_ERR_INVALID, "%s: conf / merge_mask is NULL", who);
    float *means = means_f32;
    if (!means && !(means_optional && n <= kLdsKeys)) {
        COME_REQUIRE(work != nullptr && work_bytes >= batch * n * (int64_t)sizeof(float), COME_ERR_INVALID,
                     "%s: work buffer too small (%lld bytes given)", who, (long long)work_bytes);
        means = static_cast<float *>(work);
    }
    // rank = float(threshold) * (n - 1) in fp32, as torch.quantile computes it
    const float rank = threshold * static_cast<float>(n - 1);
    int lo = static_cast<int>(std::floor(rank));
    int hi = static_cast<int>(std::ceil(rank));
    lo = lo < 0 ? 0 : (lo > n - 1 ? static_cast<int>(n - 1) : lo);
    hi = hi < 0 ? 0 : (hi > n - 1 ? static_cast<int>(n - 1) : hi);
    SelectArgs a{};
    a.conf = conf;
    a.frames = static_cast<int>(frames);
    a.H = static_cast<int>(grid_h);
    a.W = static_cast<int>(grid_w);
    a.gh = static_cast<int>(group_h);
    a.gw = static_cast<int>(group_w);
    a.mode = mode;
    a.threshold = threshold;
    a.rank_lo = lo;
    a.rank_hi = hi;
    a.frac = rank - static_cast<float>(lo);
    a.means = means;
    a.mask = merge_mask;
    a.offsets = plan ? offsets : nullptr;
    a.prefix = plan ? group_prefix : nullptr;
    a.start = static_cast<int>(start_index);
    a.post = batch == 1 ? post : nullptr;              // several batch elements: posted by the scan behind this launch
    a.post_tag = post_tag;
    a.tail = static_cast<int>(grid_h * grid_w - windows * group_h * group_w);
    a.by_windows = make_fastdiv(windows);
    a.by_mw = make_fastdiv(grid_w / group_w);
    const dim3 grid(static_cast<unsigned>(batch)), block(kSelectThreads);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool w33 = group_h == 3 && group_w == 3;
    if (mode == 0 && !plan && n <= kFewWindows) {
        const dim3 few(static_cast<unsigned>(ceil_div(n, 64) * 64));
        if (dtype == COME_BF16 && w33) hipLaunchKernelGGL((select_few_kernel<COME_BF16, 3, 3>), grid, few, 0, s, a);
        else if (dtype == COME_BF16) hipLaunchKernelGGL((select_few_kernel<COME_BF16, 0, 0>), grid, few, 0, s, a);
        else if (w33) hipLaunchKernelGGL((select_few_kernel<COME_F32, 3, 3>), grid, few, 0, s, a);
        else hipLaunchKernelGGL((select_few_kernel<COME_F32, 0, 0>), grid, few, 0, s, a);
        COME_CHECK_LAUNCH(who);
        return COME_OK;
    }
    a.given = mode != 2 && means != nullptr && n > kManyWindows && batch <= 65535;
    if (a.given) {
        const dim3 wide(static_cast<unsigned>(ceil_div(n, 256)), static_cast<unsigned>(batch));
        if (dtype == COME_BF16 && w33) hipLaunchKernelGGL((window_means_kernel<COME_BF16, 3, 3>), wide, dim3(256), 0, s, a);
        else if (dtype == COME_BF16) hipLaunchKernelGGL((window_means_kernel<COME_BF16, 0, 0>), wide, dim3(256), 0, s, a);
        else if (w33) hipLaunchKernelGGL((window_means_kernel<COME_F32, 3, 3>), wide, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((window_means_kernel<COME_F32, 0, 0>), wide, dim3(256), 0, s, a);
        COME_CHECK_LAUNCH(who);
    }
    // Few candidates are collected instead of counted again (select_kth) among fp32 means; bf16 ones are done after one or two
    // digits.
#define COME_SELECT_KEYS(DT_, GH_, GW_)                                                                                              \
    do {                                                                                                                             \
        if (n <= kSelectThreads) hipLaunchKernelGGL((select_windows_kernel<DT_, GH_, GW_, 1>), grid, block, 0, s, a);                \
        else if (n <= 4 * kSelectThreads) hipLaunchKernelGGL((select_windows_kernel<DT_, GH_, GW_, 4>), grid, block, 0, s, a);       \
        else if (n <= 8 * kSelectThreads) hipLaunchKernelGGL((select_windows_kernel<DT_, GH_, GW_, 8>), grid, block, 0, s, a);       \
        else if (n <= 16 * kSelectThreads) hipLaunchKernelGGL((select_windows_kernel<DT_, GH_, GW_, 16>), grid, block, 0, s, a);     \
        else if (n <= 32 * kSelectThreads) hipLaunchKernelGGL((select_windows_kernel<DT_, GH_, GW_, 32>), grid, block, 0, s, a);     \
        else hipLaunchKernelGGL((select_windows_kernel<DT_, GH_, GW_, 0>), grid, block, 0, s, a);                                    \
    } while (0)
    static_assert(kLdsKeys == 16 * kSelectThreads, "keys of a plan lie in LDS");
#define COME_SELECT_LAUNCH(GH_, GW_)                            \
    do {                                                        \
        if (dtype == COME_BF16) COME_SELECT_KEYS(COME_BF16, GH_, GW_); \
        else COME_SELECT_KEYS(COME_F32, GH_, GW_);              \
    } while (0)
    if (w33) COME_SELECT_LAUNCH(3, 3);
    else COME_SELECT_LAUNCH(0, 0);
#undef COME_SELECT_LAUNCH
#undef COME_SELECT_KEYS
    COME_CHECK_LAUNCH(who);
    if (plan && batch > 1) {
        hipLaunchKernelGGL(scan_offsets_kernel, dim3(1), dim3(64), 0, s, offsets, static_cast<int>(rows), post,
                           post_tag);
        COME_CHECK_LAUNCH(who);
    }
    return COME_OK;
}

}  // namespace
}  // namespace come

using namespace come;

extern "C" int64_t come_select_work_bytes(int64_t batch, int64_t frames, int64_t grid_h, int64_t grid_w,
                                          int64_t group_h, int64_t group_w) {
    if (batch < 0 || frames < 0 || grid_h < 0 || grid_w < 0 || group_h <= 0 || group_w <= 0) return -1;
    const int64_t windows = (grid_h / group_h) * (grid_w / group_w);
    return batch * frames * windows * static_cast<int64_t>(sizeof(float)) + 16;
}

extern "C" int come_select_windows(const void *conf, int dtype, int64_t batch, int64_t frames, int64_t grid_h,
                                   int64_t grid_w, int64_t group_h, int64_t group_w, int mode, float threshold,
                                   float *means_f32, uint8_t *merge_mask, void *work, int64_t work_bytes,
                                   void *stream) {
    clear_error();
    return select_impl("come_select_windows", conf, dtype, batch, frames, grid_h, grid_w, group_h, group_w, mode,
                       threshold, means_f32, merge_mask, work, work_bytes, false, 0, nullptr, nullptr, stream);
}

extern "C" int come_select_plan(const void *conf, int dtype, int64_t batch, int64_t frames, int64_t grid_h,
                                int64_t grid_w, int64_t group_h, int64_t group_w, int mode, float threshold,
                                int64_t start_index, float *means_f32, uint8_t *merge_mask, int32_t *offsets,
                                int32_t *group_prefix, void *work, int64_t work_bytes, void *stream) {
    clear_error();
    return select_impl("come_select_plan", conf, dtype, batch, frames, grid_h, grid_w, group_h, group_w, mode,
                       threshold, means_f32, merge_mask, work, work_bytes, true, start_index, offsets, group_prefix,
                       stream);
}

extern "C" int come_select_plan_post(const void *conf, int dtype, int64_t batch, int64_t frames, int64_t grid_h,
                                     int64_t grid_w, int64_t group_h, int64_t group_w, int mode, float threshold,
                                     int64_t start_index, float *means_f32, uint8_t *merge_mask, int32_t *offsets,
                                     int32_t *group_prefix, void *work, int64_t work_bytes, uint64_t *post,
                                     uint32_t tag, void *stream) {
    clear_error();
    return select_impl("come_select_plan_post", conf, dtype, batch, frames, grid_h, grid_w, group_h, group_w, mode,
                       threshold, means_f32, merge_mask, work, work_bytes, true, start_index, offsets, group_prefix,
                       stream, true, post, tag);
}
