// Token merge / unmerge for gfx950: HBM-bound gather-mean and gather kernels.
//
// Data movement is organised in 16-byte chunks: one thread owns one chunk column of
// one window (or of one copied token), issues all of the window's loads back to back
// (nine independent 16-byte loads for a 3x3 window) and writes either their mean
// (merged) or the rows themselves (kept).  A wavefront therefore reads 1 KiB
// contiguous per source row and writes 1 KiB contiguous per packed row.  Token data is
// touched once, so loads and stores carry the non-temporal hint; the rows an unmerge
// reads several times (merged windows) use ordinary loads and stay in L2.
#include "come_common.h"

#include <algorithm>
#include <type_traits>

namespace come {
namespace {

constexpr int kThreads = 256;
// the 16-byte merge kernel runs one wavefront per workgroup (measured at 64 / 128 / 256 / 512 / 1024 threads on the
// 16-frame microbenchmark: 14.2 / 14.6 / 14.8 / 16.0 / 18.1 us)
constexpr int kMergeThreads = 64;

struct MergeGeom {
    int rows, n_tok, start, groups;
    int gh, gw, G;          // window shape, tokens per window
    int H, W, mw;           // token grid, windows per grid row
    int cov_h, cov_w;       // part of the grid covered by full windows
    int tail;               // grid positions outside the full windows
    int64_t out_rows;
};

struct MergeArgs {
    MergeGeom g;
    const void *tokens;
    void *out;
    const uint8_t *mask;
    const int32_t *offsets;
    const int32_t *prefix;
    int64_t *rev64;
    int32_t *rev32;
    float *weight;
    int32_t *count;
    int64_t *offsets64;      // optional: the row offsets once more, widened
    int64_t group_items;     // rows * groups * chunks (or * chans in the scalar kernel)
    int64_t group_blocks;    // blocks that own group items
    int64_t single_items;    // rows * (start + tail) * chunks
    int chunks;              // 16-byte chunks per token row (vector kernel) / chans (scalar kernel)
    FastDiv by_chunks, by_groups, by_mw, by_per_row, by_side;   // 16-byte kernels only
    uint64_t *post;          // DIRECT: where the packed row count goes as soon as it is known (optional), with post_tag
    uint32_t post_tag;
};

__device__ inline void note_row(const MergeArgs &a, int64_t src_flat, int64_t dst) {
    if (a.rev64) a.rev64[src_flat] = dst;
    if (a.rev32) a.rev32[src_flat] = static_cast<int32_t>(dst);
}
__device__ inline void note_weight(const MergeArgs &a, int64_t dst, int n) {
    if (dst >= a.g.out_rows) return;
    if (a.weight) a.weight[dst] = static_cast<float>(n);
    if (a.count) a.count[dst] = n;
}

// A mask byte per window, four to a word: how many are set / which (bit i: byte i).
__device__ inline uint32_t set_bytes(uint32_t w) { return (((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w) & 0x80808080u; }
__device__ inline int nonzero_bytes(uint32_t w) { return __popc(set_bytes(w)); }
__device__ inline uint32_t nonzero_bits(uint32_t w) { return ((set_bytes(w) >> 7) * 0x01020408u) >> 24; }

// ---------------------------------------------------------------------------------
// Merging straight from the mask (DIRECT kernels).  With C(n) the number of merged windows among the first n of the flat
// mask, every packed position has a closed form: what lies at position t of its row's dense order (specials, windows,
// leftover) moves from b * n_tok + t to b * n_tok + t - (G - 1) * C(windows in front of it).  A wavefront counts the
// mask in front of its own window itself, 16 bytes per lane and step, while its token loads are on their way; one
// workgroup in front of the others counts all of it and posts the packed row count.  That saves the plan launch in front of
// a merge (2.2 - 3.4 us and the gap behind it) wherever the size of the outputs is known beforehand: confidence -> packed
// tokens and positions 28.9 -> 26.2 us (1 frame of 80 windows), 39.0 -> 34.0 (16 frames of 144), 53 -> 48.8 (32 frames),
// 82 -> 79.6 (64).  The reads of the mask grow with the square of its size, and what there is to gain stays the same: 113
// frames (16 272 windows) 128.1 -> 127.5.  Larger masks are planned, and light windows from half of that on (come_token_merge_is_direct).
// ---------------------------------------------------------------------------------
constexpr int kDirectWindows = 16384;
constexpr int kMaskAhead = 4;            // 16-byte loads of the mask per lane in front of the token loads (4096 windows)

struct MaskCount {
    uint4 w[kMaskAhead];
    __device__ inline void request(const uint8_t *mask, uint32_t n, int lane) {              // n: wave-uniform
#pragma unroll
        for (int s = 0; s < kMaskAhead; ++s) {
            w[s] = make_uint4(0, 0, 0, 0);
            const uint32_t i = static_cast<uint32_t>(lane) + 64u * s;
            if (i < n / 16) w[s] = reinterpret_cast<const uint4 *>(mask)[i];
        }
    }
    // merged windows among the first n - n % 16
    __device__ inline int total(const uint8_t *mask, uint32_t n, int lane) const {
        int count = 0;
#pragma unroll
        for (int s = 0; s < kMaskAhead; ++s) count += nonzero_bytes(w[s].x) + nonzero_bytes(w[s].y) + nonzero_bytes(w[s].z) + nonzero_bytes(w[s].w);
        for (uint32_t i = static_cast<uint32_t>(lane) + 64u * kMaskAhead; i < n / 16; i += 64) {
            const uint4 v = reinterpret_cast<const uint4 *>(mask)[i];
            count += nonzero_bytes(v.x) + nonzero_bytes(v.y) + nonzero_bytes(v.z) + nonzero_bytes(v.w);
        }
        return __builtin_amdgcn_readlane(static_cast<int>(wave_scan_add(static_cast<uint32_t>(count))), 63);
    }
};

// which of the windows [n - n % 16, + 64) are merged, bit by bit (all lanes of the wavefront take part)
__device__ inline uint64_t mask_bits_at(const uint8_t *mask, uint32_t n, uint32_t windows, int lane) {
    const uint32_t i = (n & ~15u) + static_cast<uint32_t>(lane);
    return __ballot(i < windows && mask[i] != 0);
}
__device__ inline int bits_below(uint64_t bits, uint32_t n) { return __popcll(bits & ((1ull << n) - 1ull)); }      // n < 64

// offsets64[0 .. rows] <- offsets[0 .. rows], spread over the launch
__device__ inline void widen_offsets(const MergeArgs &a) {
    if (a.offsets64 == nullptr) return;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i <= a.g.rows;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x)
        a.offsets64[i] = a.offsets[i];
}

// position `r` (0-based) among the grid positions outside the full windows, image row-major
__device__ inline int leftover_position(const MergeGeom &g, int r) {
    const int side = g.W - g.cov_w;                 // leftover columns of a covered grid row
    const int upper = g.cov_h * side;
    if (r < upper) {
        const int y = r / side;
        return y * g.W + g.cov_w + (r - y * side);
    }
    return g.cov_h * g.W + (r - upper);
}

__device__ inline int leftover_position_fast(const MergeGeom &g, const FastDiv &by_side, int r) {
    const int side = g.W - g.cov_w;
    const int upper = g.cov_h * side;
    if (r < upper) {
        const int y = static_cast<int>(fast_div(static_cast<uint32_t>(r), by_side));
        return y * g.W + g.cov_w + (r - y * side);
    }
    return g.cov_h * g.W + (r - upper);
}

// ---------------------------------------------------------------------------------
// bookkeeping: mask -> per-window prefix, per-row length, row offsets.  A wavefront owns a row; up to
// kPlanRowsPerGroup rows run as one workgroup that also scans the lengths, more rows are spread
// over workgroups and a one-wavefront launch scans afterwards.
// ---------------------------------------------------------------------------------
constexpr int kPlanRowsPerGroup = 16;

__device__ inline int scan_row_lengths(int32_t *__restrict__ offsets, int rows) {   // one wavefront, in place; the total
    const int lane = threadIdx.x & 63;
    int carry = 0;
    for (int r0 = 0; r0 < rows; r0 += 64) {
        const int r = r0 + lane;
        int v = r < rows ? offsets[r + 1] : 0;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int t = __shfl_up(v, d);
            if (lane >= d) v += t;
        }
        if (r < rows) offsets[r + 1] = v + carry;
        carry += __shfl(v, 63);
    }
    return carry;
}

__global__ __launch_bounds__(64 * kPlanRowsPerGroup) void merge_plan_kernel(const uint8_t *__restrict__ mask, int rows,
                                                                            int groups, int start, int G, int tail,
                                                                            int32_t *__restrict__ offsets,
                                                                            int32_t *__restrict__ prefix, uint64_t *post,
                                                                            uint32_t post_tag) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const uint64_t below = (1ull << lane) - 1ull;

    for (int b = blockIdx.x * kPlanRowsPerGroup + wave; b < rows; b += gridDim.x * kPlanRowsPerGroup) {
        int running = 0;                                    // wave-uniform
        for (int m0 = 0; m0 < groups; m0 += 64) {
            const int m = m0 + lane;
            const bool valid = m < groups;
            const bool merged = valid && mask[static_cast<int64_t>(b) * groups + m] != 0;
            const uint64_t merged_bits = __ballot(merged);
            const int merged_before = __popcll(merged_bits & below);
            if (valid) prefix[static_cast<int64_t>(b) * groups + m] = running + merged_before + (lane - merged_before) * G;
            const int n_valid = min(64, groups - m0);
            const int n_merged = __popcll(merged_bits);
            running += n_merged + (n_valid - n_merged) * G;
        }
        if (lane == 0) offsets[b + 1] = start + tail + running;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) offsets[0] = 0;
    if (gridDim.x > 1) return;                              // the scan is the next launch
    __syncthreads();
    if (wave != 0) return;
    const int total = scan_row_lengths(offsets, rows);
    if (post != nullptr && lane == 0) post_to_host(post, post_tag, static_cast<uint32_t>(total));
}

__global__ __launch_bounds__(64) void merge_plan_scan_kernel(int32_t *__restrict__ offsets, int rows, uint64_t *post,
                                                             uint32_t post_tag) {
    const int total = scan_row_lengths(offsets, rows);
    if (post != nullptr && threadIdx.x == 0) post_to_host(post, post_tag, static_cast<uint32_t>(total));
}

// The same plan in one launch without a scan behind it: a workgroup per row counts the merged windows of all rows in
// front of its own by itself (16 mask bytes per lane and step), which gives its row's offset in closed form.  Reads of
// the mask grow with the square of the row count, so this form takes masks whose workgroups together read at most
// kPlanRescanBytes (128 rows of 144 windows: 1.2 MB out of L2).  32 rows of 1024 groups: 5.2 us, against 7.5 + 5.3 us of
// the two launches that more rows take.
constexpr int kPlanThreads = 256;
constexpr int64_t kPlanRescanBytes = 16 << 20;

__global__ __launch_bounds__(kPlanThreads) void merge_plan_rows_kernel(const uint8_t *__restrict__ mask, int rows, int groups,
                                                                       int start, int G, int tail,
                                                                       int32_t *__restrict__ offsets,
                                                                       int32_t *__restrict__ prefix, uint64_t *post,
                                                                       uint32_t post_tag) {
    constexpr int kWaves = kPlanThreads / 64;
    __shared__ int lds_count[kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    const int b = blockIdx.x;
    const int before = b * groups;                                          // mask bytes in front of this row
    int count = 0;
    for (int i = threadIdx.x; i < before / 16; i += kPlanThreads) {
        const uint4 w = reinterpret_cast<const uint4 *>(mask)[i];
        count += nonzero_bytes(w.x) + nonzero_bytes(w.y) + nonzero_bytes(w.z) + nonzero_bytes(w.w);
    }
    if (static_cast<int>(threadIdx.x) < before % 16) count += mask[before - before % 16 + threadIdx.x] != 0 ? 1 : 0;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) count += __shfl_xor(count, d);
    if (lane == 0) lds_count[wave] = count;
    __syncthreads();
    int merged_in_front = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) merged_in_front += lds_count[w];
    int merged = 0;                                                         // of this row, so far (uniform)
    for (int m0 = 0; m0 < groups; m0 += kPlanThreads) {
        const int m = m0 + threadIdx.x;
        const bool is_merged = m < groups && mask[before + m] != 0;
        const uint64_t bits = __ballot(is_merged);
        __syncthreads();                                                    // the counts of the step before have been read
        if (lane == 0) lds_count[wave] = __popcll(bits);
        __syncthreads();
        int mine = merged + __popcll(bits & below);
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            mine += w < wave ? lds_count[w] : 0;
            merged += lds_count[w];
        }
        if (m < groups) prefix[before + m] = m * G - mine * (G - 1);
    }
    if (threadIdx.x == 0) {
        const int full = start + tail + groups * G;                         // length of a row that merges nothing
        const int end = (b + 1) * full - (merged_in_front + merged) * (G - 1);
        if (b == 0) offsets[0] = 0;
        offsets[b + 1] = end;
        if (post != nullptr && b == rows - 1) post_to_host(post, post_tag, static_cast<uint32_t>(end));
    }
}

// ---------------------------------------------------------------------------------
// merge, 16-byte path.  GH x GW fixed at compile time (0 x 0 = run-time window shape).  DIRECT: without a plan (at least two
// chunks a row, so that a wavefront's windows lie within the 64 whose bits it looks at).
// ---------------------------------------------------------------------------------
template <int DT, int GH, int GW, bool DIRECT>
__global__ __launch_bounds__(kMergeThreads) void merge_vec_kernel(const MergeArgs a) {
    static_assert(kMergeThreads == 64, "a workgroup is a wavefront");
    using V = Vec16<DT>;
    const MergeGeom &g = a.g;
    const uint4 *__restrict__ src = static_cast<const uint4 *>(a.tokens);
    uint4 *__restrict__ dst = static_cast<uint4 *>(a.out);
    const int chunks = a.chunks;
    const int lane = threadIdx.x;
    const uint32_t windows = static_cast<uint32_t>(g.rows) * static_cast<uint32_t>(g.groups);      // (of this launch)
    uint32_t block = blockIdx.x;
    if constexpr (DIRECT) {
        if (block == 0) {                                   // the packed row count
            MaskCount ahead;
            ahead.request(a.mask, windows, lane);
            const uint64_t bits = mask_bits_at(a.mask, windows, windows, lane);
            const int merged = ahead.total(a.mask, windows, lane) + __popcll(bits);
            const int rows = g.rows * g.n_tok - (g.G - 1) * merged;
            if (lane == 0) {
                if (a.post != nullptr) post_to_host(a.post, a.post_tag, static_cast<uint32_t>(rows));
                if (a.offsets64 != nullptr) a.offsets64[g.rows] = rows;
            }
            return;
        }
        --block;
    } else {
        widen_offsets(a);
    }

    if (static_cast<int64_t>(block) < a.group_blocks) {
        const uint32_t id0 = block * kMergeThreads;
        uint32_t id = id0 + threadIdx.x;                    // item counts stay below 2^31 (checked by the host)
        const bool inside = id < a.group_items;
        MaskCount ahead;
        uint64_t bits = 0;                                  // windows from base on
        uint32_t gm0 = 0;
        if constexpr (DIRECT) {
            gm0 = __builtin_amdgcn_readfirstlane(fast_div(id0, a.by_chunks));
            ahead.request(a.mask, gm0, lane);
            bits = mask_bits_at(a.mask, gm0, windows, lane);
            if (!inside) id = id0;                          // (every lane counts)
        } else {
            if (!inside) return;
        }
        const uint32_t gm = fast_div(id, a.by_chunks);      // flat (row, window)
        const int chunk = static_cast<int>(id - gm * chunks);
        const int b = static_cast<int>(fast_div(gm, a.by_groups));
        const int m = static_cast<int>(gm) - b * g.groups;
        const int wy = static_cast<int>(fast_div(m, a.by_mw));
        const int wx = m - wy * g.mw;
        bool merged;
        int64_t row0;
        if constexpr (DIRECT) {
            merged = (bits >> (gm - (gm0 & ~15u))) & 1;
        } else {
            merged = a.mask[gm] != 0;
            row0 = static_cast<int64_t>(a.offsets[b]) + g.start + a.prefix[gm];
        }
        const int64_t tok0 = static_cast<int64_t>(b) * g.n_tok + g.start + (wy * g.gh) * g.W + wx * g.gw;
        const uint4 *p = src + tok0 * chunks + chunk;
        // DIRECT: behind the token loads
        auto place = [&]() __attribute__((always_inline)) {
            if constexpr (DIRECT) {
                const int before = ahead.total(a.mask, gm0, lane) + bits_below(bits, gm - (gm0 & ~15u));
                row0 = static_cast<int64_t>(b) * g.n_tok + g.start + m * g.G - static_cast<int64_t>(g.G - 1) * before;
                if (inside && m == 0 && chunk == 0 && a.offsets64 != nullptr) a.offsets64[b] = row0 - g.start;
            }
        };

        if constexpr (GH > 0) {
            uint4 v[GH * GW];
#pragma unroll
            for (int dy = 0; dy < GH; ++dy)
#pragma unroll
                for (int dx = 0; dx < GW; ++dx)
                    v[dy * GW + dx] = ld16_stream(p + (static_cast<int64_t>(dy) * g.W + dx) * chunks);
            place();
            if (DIRECT && !inside) return;
            if (merged) {
                float acc[V::N];
#pragma unroll
                for (int e = 0; e < V::N; ++e) acc[e] = 0.f;
#pragma unroll
                for (int t = 0; t < GH * GW; ++t) {
                    float f[V::N];
                    V::unpack(v[t], f);
#pragma unroll
                    for (int e = 0; e < V::N; ++e) acc[e] += f[e];
                }
#pragma unroll
                for (int e = 0; e < V::N; ++e) acc[e] = acc[e] / static_cast<float>(GH * GW);
                if (row0 < g.out_rows) st16_stream(dst + row0 * chunks + chunk, V::pack(acc));
            } else {
#pragma unroll
                for (int t = 0; t < GH * GW; ++t)
                    if (row0 + t < g.out_rows) st16_stream(dst + (row0 + t) * chunks + chunk, v[t]);
            }
        } else {
            place();
            if (DIRECT && !inside) return;
            if (merged) {
                float acc[V::N];
#pragma unroll
                for (int e = 0; e < V::N; ++e) acc[e] = 0.f;
                for (int dy = 0; dy < g.gh; ++dy) {
#pragma unroll 4
                    for (int dx = 0; dx < g.gw; ++dx) {
                        float f[V::N];
                        V::unpack(p[(static_cast<int64_t>(dy) * g.W + dx) * chunks], f);
#pragma unroll
                        for (int e = 0; e < V::N; ++e) acc[e] += f[e];
                    }
                }
#pragma unroll
                for (int e = 0; e < V::N; ++e) acc[e] = acc[e] / static_cast<float>(g.G);
                if (row0 < g.out_rows) dst[row0 * chunks + chunk] = V::pack(acc);
            } else {
                int64_t r = row0;
                for (int dy = 0; dy < g.gh; ++dy) {
#pragma unroll 4
                    for (int dx = 0; dx < g.gw; ++dx, ++r)
                        if (r < g.out_rows) dst[r * chunks + chunk] = p[(static_cast<int64_t>(dy) * g.W + dx) * chunks];
                }
            }
        }

        // index map and counts of this window: token t of the window is noted by the thread of chunk t, so the
        // few small stores go out side by side instead of one after the other from a single lane
        const int gw_rt = GH > 0 ? GW : g.gw;
        for (int t = chunk; t < g.G; t += chunks) {
            const int dy = t / gw_rt;
            const int dx = t - dy * gw_rt;
            note_row(a, tok0 + static_cast<int64_t>(dy) * g.W + dx, merged ? row0 : row0 + t);
            if (!merged) note_weight(a, row0 + t, 1);
        }
        if (merged && chunk == 0) note_weight(a, row0, g.G);
        return;
    }

    // copied tokens: specials in front, leftover grid positions behind the windows
    uint32_t id = (block - static_cast<uint32_t>(a.group_blocks)) * kMergeThreads + threadIdx.x;
    const bool inside = id < a.single_items;
    if (!inside) {
        if constexpr (!DIRECT) return;
        id -= threadIdx.x;                                  // (every lane counts)
    }
    const int per_row = g.start + g.tail;
    const uint32_t t = fast_div(id, a.by_chunks);
    const int chunk = static_cast<int>(id - t * chunks);
    const int b = static_cast<int>(fast_div(t, a.by_per_row));
    const int j = static_cast<int>(t) - b * per_row;
    int64_t flat, row;
    if constexpr (DIRECT) {
        const int r = j - g.start;
        flat = static_cast<int64_t>(b) * g.n_tok + (j < g.start ? j : g.start + leftover_position_fast(g, a.by_side, r));
        const uint4 v = ld16_stream(src + flat * chunks + chunk);
        const uint32_t front = static_cast<uint32_t>(j < g.start ? b : b + 1) * static_cast<uint32_t>(g.groups);     // windows in front
        // The fronts rise with the lanes, by a row's windows from one row to the next: one count up to the first of them, the rest
        // from the mask behind it, 1024 windows a step.  (A count for each of up to 32 rows took 53 us for 512 rows of 65 tokens of
        // 32 bytes, 16 384 windows; the plan and a merge behind it take 11.)
        const uint32_t n0 = __builtin_amdgcn_readfirstlane(front);
        const uint32_t n1 = __builtin_amdgcn_readlane(front, 63 - __builtin_clzll(__ballot(inside)));
        const uint32_t whole = windows / 16;
        auto step_of = [&](uint32_t c0) __attribute__((always_inline)) {
            const uint32_t i = c0 + static_cast<uint32_t>(lane);
            return i < whole ? reinterpret_cast<const uint4 *>(a.mask)[i] : make_uint4(0, 0, 0, 0);
        };
        MaskCount ahead;
        ahead.request(a.mask, n0, lane);
        uint4 next = make_uint4(0, 0, 0, 0);
        uint32_t last = 0;                                  // of chunk `whole`
        if ((n0 & ~15u) < n1) {
            next = step_of(n0 / 16);
            if (16 * whole < n1) last = static_cast<uint32_t>(mask_bits_at(a.mask, windows, windows, lane)) & 0xffffu;
        }
        int before = ahead.total(a.mask, n0, lane);
        for (uint32_t c0 = n0 / 16; 16 * c0 < n1; c0 += 64) {
            const uint4 w = next;
            next = step_of(c0 + 64);
            uint32_t bits = nonzero_bits(w.x) | nonzero_bits(w.y) << 4 | nonzero_bits(w.z) << 8 | nonzero_bits(w.w) << 12;
            if (c0 + static_cast<uint32_t>(lane) == whole) bits = last;
            const int upto = static_cast<int>(wave_scan_add(static_cast<uint32_t>(__popc(bits))));
            const int all = __builtin_amdgcn_readlane(upto, 63);                                  // (with every lane active)
            const int own = static_cast<int>(front / 16) - static_cast<int>(c0);                 // the lane that holds this one's front
            const int from = min(max(own, 0), 63);
            const int theirs = __shfl(upto, from);
            const uint32_t chunk_bits = __shfl(bits, from);
            if (own >= 64) before += all;
            else if (own >= 0) before += theirs - __popc(chunk_bits) + __popc(chunk_bits & ((1u << (front & 15u)) - 1u));
        }
        if (!inside) return;
        row = (j < g.start ? flat : static_cast<int64_t>(b + 1) * g.n_tok - g.tail + r) - static_cast<int64_t>(g.G - 1) * before;
        if (row < g.out_rows) st16_stream(dst + row * chunks + chunk, v);
    } else {
        int tok;
        if (j < g.start) {
            tok = j;
            row = static_cast<int64_t>(a.offsets[b]) + j;
        } else {
            const int r = j - g.start;
            tok = g.start + leftover_position_fast(g, a.by_side, r);
            row = static_cast<int64_t>(a.offsets[b + 1]) - g.tail + r;
        }
        flat = static_cast<int64_t>(b) * g.n_tok + tok;
        if (row < g.out_rows) st16_stream(dst + row * chunks + chunk, ld16_stream(src + flat * chunks + chunk));
    }
    if (chunk == 0) {
        note_row(a, flat, row);
        note_weight(a, row, 1);
    }
}

// ---------------------------------------------------------------------------------
// merge, element path: any channel count / alignment (e.g. the 2-channel position
// tensor).  One thread per (window, channel) or (copied token, channel).
// ---------------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(kThreads) void merge_elem_kernel(const MergeArgs a) {
    using V = Vec16<DT>;
    const MergeGeom &g = a.g;
    const int chans = a.chunks;
    widen_offsets(a);

    if (static_cast<int64_t>(blockIdx.x) < a.group_blocks) {
        const int64_t id = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
        if (id >= a.group_items) return;
        const int64_t gm = id / chans;
        const int c = static_cast<int>(id - gm * chans);
        const int b = static_cast<int>(gm / g.groups);
        const int m = static_cast<int>(gm - static_cast<int64_t>(b) * g.groups);
        const int wy = m / g.mw;
        const int wx = m - wy * g.mw;
        const bool merged = a.mask[gm] != 0;
        const int64_t row0 = static_cast<int64_t>(a.offsets[b]) + g.start + a.prefix[gm];
        const int64_t tok0 = static_cast<int64_t>(b) * g.n_tok + g.start + (wy * g.gh) * g.W + wx * g.gw;
        float acc = 0.f;
        int t = 0;
        for (int dy = 0; dy < g.gh; ++dy) {
            for (int dx = 0; dx < g.gw; ++dx, ++t) {
                const int64_t tok = tok0 + static_cast<int64_t>(dy) * g.W + dx;
                const float x = V::load1(a.tokens, tok * chans + c);
                if (merged) {
                    acc += x;
                } else if (row0 + t < g.out_rows) {
                    V::store1(a.out, (row0 + t) * chans + c, x);
                }
                if (c == 0) {
                    note_row(a, tok, merged ? row0 : row0 + t);
                    if (!merged) note_weight(a, row0 + t, 1);
                }
            }
        }
        if (merged) {
            if (row0 < g.out_rows) V::store1(a.out, row0 * chans + c, acc / static_cast<float>(g.G));
            if (c == 0) note_weight(a, row0, g.G);
        }
        return;
    }

    const int64_t id = (static_cast<int64_t>(blockIdx.x) - a.group_blocks) * kThreads + threadIdx.x;
    if (id >= a.single_items) return;
    const int per_row = g.start + g.tail;
    const int64_t t = id / chans;
    const int c = static_cast<int>(id - t * chans);
    const int b = static_cast<int>(t / per_row);
    const int j = static_cast<int>(t - static_cast<int64_t>(b) * per_row);
    int tok;
    int64_t row;
    if (j < g.start) {
        tok = j;
        row = static_cast<int64_t>(a.offsets[b]) + j;
    } else {
        const int r = j - g.start;
        tok = g.start + leftover_position(g, r);
        row = static_cast<int64_t>(a.offsets[b + 1]) - g.tail + r;
    }
    const int64_t flat = static_cast<int64_t>(b) * g.n_tok + tok;
    if (row < g.out_rows) V::store1(a.out, row * chans + c, V::load1(a.tokens, flat * chans + c));
    if (c == 0) {
        note_row(a, flat, row);
        note_weight(a, row, 1);
    }
}

// ---------------------------------------------------------------------------------
// merge of narrow rows (at most kNarrowChans channels: the position tensors).  One thread per dense token, whatever
// its kind: index map entries go out coalesced, a kept token is one independent load and store, and only the first
// token of a merged window walks the window (its reads hit the lines its neighbours fetch).  The launch is a handful
// of microseconds of dependent latency, not bytes: the element kernel's serial walk of every window by one thread took
// 5.6 us for 16 frames of 37 x 37, this one 3.9 us.
// ---------------------------------------------------------------------------------
// DIRECT: every workgroup counts the whole mask into LDS first, 16 windows to an entry (merged windows in front of the 16
// in the high bits, the 16 themselves in the low ones).
// ---------------------------------------------------------------------------------
constexpr int kNarrowChans = 4;

struct MaskTable {
    static constexpr int kPer = kDirectWindows / 16 / kThreads;            // entries per thread
    uint32_t entry[kDirectWindows / 16 + 1];
    uint32_t waves[kThreads / 64];
    __device__ inline int before(uint32_t n) const {                       // C(n), n up to and with the number of windows
        const uint32_t e = entry[n >> 4];
        return static_cast<int>(e >> 16) + __popc(e & ((1u << (n & 15u)) - 1u));
    }
    __device__ inline bool merged(uint32_t n) const { return (entry[n >> 4] >> (n & 15u)) & 1u; }
    __device__ inline void fill(const uint8_t *mask, uint32_t windows) {
        uint32_t bits[kPer];
        const uint32_t used = (windows + 16 * kThreads - 1) / (16 * kThreads);         // entries a thread has to look at (uniform)
#pragma unroll
        for (uint32_t s = 0; s < kPer; ++s) {
            bits[s] = 0;
            if (s >= used) continue;
            const uint32_t at = 16 * (threadIdx.x * used + s);
            if (at + 16 <= windows) {
                const uint4 w = *reinterpret_cast<const uint4 *>(mask + at);
                bits[s] = nonzero_bits(w.x) | (nonzero_bits(w.y) << 4) | (nonzero_bits(w.z) << 8) | (nonzero_bits(w.w) << 12);
            } else if (at < windows) {
                for (uint32_t i = 0; i < windows - at; ++i) bits[s] |= (mask[at + i] != 0 ? 1u : 0u) << i;
            }
        }
        uint32_t mine = 0;
#pragma unroll
        for (uint32_t s = 0; s < kPer; ++s) mine += __popc(bits[s]);
        const uint32_t upto = wave_scan_add(mine);
        if ((threadIdx.x & 63) == 63) waves[threadIdx.x >> 6] = upto;
        __syncthreads();
        uint32_t run = upto - mine;
#pragma unroll
        for (uint32_t w = 0; w < kThreads / 64; ++w) run += w < (threadIdx.x >> 6) ? waves[w] : 0;
#pragma unroll
        for (uint32_t s = 0; s < kPer; ++s) {
            if (s >= used) continue;
            entry[threadIdx.x * used + s] = (run << 16) | bits[s];
            run += __popc(bits[s]);
        }
        if (threadIdx.x == kThreads - 1) entry[kThreads * used] = run << 16;
        __syncthreads();
    }
};

template <int DT, int CH, bool DIRECT>
__global__ __launch_bounds__(kThreads) void merge_narrow_kernel(const MergeArgs a) {
    using V = Vec16<DT>;
    const MergeGeom &g = a.g;
    __shared__ std::conditional_t<DIRECT, MaskTable, char> table;
    const uint32_t flat = blockIdx.x * kThreads + threadIdx.x;             // rows * n_tok < 2^31 (checked by the host)
    if constexpr (DIRECT) {
        const uint32_t windows = static_cast<uint32_t>(g.rows) * static_cast<uint32_t>(g.groups);
        table.fill(a.mask, windows);
        if (flat == 0) {
            const int rows = g.rows * g.n_tok - (g.G - 1) * table.before(windows);
            if (a.post != nullptr) post_to_host(a.post, a.post_tag, static_cast<uint32_t>(rows));
            if (a.offsets64 != nullptr) a.offsets64[g.rows] = rows;
        }
    } else {
        widen_offsets(a);
    }
    if (flat >= a.group_items) return;
    const int b = static_cast<int>(fast_div(flat, a.by_groups));           // by tokens per row
    const int tok = static_cast<int>(flat) - b * g.n_tok;
    const int p = tok - g.start;
    const int y = p < 0 ? 0 : static_cast<int>(fast_div(static_cast<uint32_t>(p), a.by_per_row));   // by the grid's width
    const int x = p - y * g.W;
    auto before = [&](uint32_t n) __attribute__((always_inline)) {
        if constexpr (DIRECT) return table.before(n);
        else return 0;
    };
    auto is_merged = [&](uint32_t n) __attribute__((always_inline)) {
        if constexpr (DIRECT) return table.merged(n);
        else return a.mask[n] != 0;
    };
    int64_t row;                                                            // in front of the merges before it (DIRECT) or after them
    uint32_t front = static_cast<uint32_t>(b) * static_cast<uint32_t>(g.groups);      // windows in front of it
    int merged_t = -1;                                                      // position inside a merged window
    if constexpr (DIRECT) row = flat;
    else row = p < 0 ? static_cast<int64_t>(a.offsets[b]) + tok : 0;
    if (DIRECT && tok == 0 && a.offsets64 != nullptr) a.offsets64[b] = row - static_cast<int64_t>(g.G - 1) * before(front);
    if (p >= 0 && y < g.cov_h && x < g.cov_w) {
        const int wy = static_cast<int>(fast_div(static_cast<uint32_t>(y), a.by_chunks));           // by the window's height
        const int wx = static_cast<int>(fast_div(static_cast<uint32_t>(x), a.by_mw));               // by the window's width
        const int m = wy * g.mw + wx;
        front += m;
        const int t = (y - wy * g.gh) * g.gw + (x - wx * g.gw);
        if constexpr (DIRECT) row = static_cast<int64_t>(b) * g.n_tok + g.start + m * g.G;
        else row = static_cast<int64_t>(a.offsets[b]) + g.start + a.prefix[front];
        if (is_merged(front)) merged_t = t;
        else row += t;
    } else if (p >= 0) {
        const int side = g.W - g.cov_w;
        const int r = y < g.cov_h ? y * side + (x - g.cov_w) : g.cov_h * side + (y - g.cov_h) * g.W + x;
        front += g.groups;
        if constexpr (DIRECT) row = static_cast<int64_t>(b + 1) * g.n_tok - g.tail + r;
        else row = static_cast<int64_t>(a.offsets[b + 1]) - g.tail + r;
    }
    if constexpr (DIRECT) row -= static_cast<int64_t>(g.G - 1) * before(front);
    note_row(a, flat, row);
    if (merged_t > 0 || row >= g.out_rows) return;
    float acc[CH];
    if (merged_t < 0) {
#pragma unroll
        for (int c = 0; c < CH; ++c) acc[c] = V::load1(a.tokens, static_cast<int64_t>(flat) * CH + c);
#pragma unroll
        for (int c = 0; c < CH; ++c) V::store1(a.out, row * CH + c, acc[c]);
        note_weight(a, row, 1);
        return;
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) acc[c] = 0.f;
    for (int dy = 0; dy < g.gh; ++dy)
#pragma unroll 4
        for (int dx = 0; dx < g.gw; ++dx)
#pragma unroll
            for (int c = 0; c < CH; ++c)
                acc[c] += V::load1(a.tokens, (static_cast<int64_t>(flat) + static_cast<int64_t>(dy) * g.W + dx) * CH + c);
#pragma unroll
    for (int c = 0; c < CH; ++c) V::store1(a.out, row * CH + c, acc[c] / static_cast<float>(g.G));
    note_weight(a, row, g.G);
}

// ---------------------------------------------------------------------------------
// unmerge: out[i, :] = merged[rev[i], :]
// ---------------------------------------------------------------------------------
// Output rows that stay on one XCD.  What outgrows the Infinity Cache runs in shorter ones: 128 frames of 1226 rows, fp32, 1024
// channels 158.3 -> 154.5 us, the pair of them 320 -> 312; smaller ones are slower for it (48 frames, bf16 27.7 -> 29.0).
constexpr int kSplitRunRows = 256, kSplitRunRowsLarge = 64;
constexpr int64_t kSplitLarge = 256ll << 20;          // bytes read and written

// PAIR: two packed sources with one index map; an output row holds the row of `merged` followed by the row of
// `merged_b` (`chunks` is the width of one source row, an output row has 2 * chunks chunks).
template <typename IndexT, bool PAIR>
__global__ __launch_bounds__(kThreads) void split_vec_kernel(const uint4 *__restrict__ merged,
                                                             const uint4 *__restrict__ merged_b, int64_t merged_rows,
                                                             const IndexT *__restrict__ rev, int chunks,
                                                             uint4 *__restrict__ out, int64_t items,
                                                             FastDiv by_out_chunks, uint32_t run) {
    // workgroup i runs on XCD i % 8; dealing the output rows to the XCDs in runs of `run` consecutive workgroups
    // (kSplitRunRows output rows) keeps the (up to nine) consumers of a merged row on one L2
    uint32_t bid = blockIdx.x;
    if (bid < (gridDim.x / (8u * run)) * (8u * run)) {
        const uint32_t local = bid >> 3;
        bid = ((local / run) * 8u + (bid & 7u)) * run + local % run;
    }
    const uint32_t id = bid * kThreads + threadIdx.x;               // items < 2^31 (checked by the host)
    if (id >= items) return;
    const int out_chunks = PAIR ? 2 * chunks : chunks;
    const uint32_t row = fast_div(id, by_out_chunks);
    const int out_chunk = static_cast<int>(id - row * out_chunks);
    const bool second = PAIR && out_chunk >= chunks;
    const uint4 *__restrict__ src = second ? merged_b : merged;
    const int chunk = second ? out_chunk - chunks : out_chunk;
    const int64_t from = static_cast<int64_t>(rev[row]);
    uint4 v = make_uint4(0, 0, 0, 0);
    if (from >= 0 && from < merged_rows) v = src[from * chunks + chunk];
    st16_stream(out + id, v);
}

// Wave-per-row form for rows that are a multiple of 1 KiB wide (64 chunks): a wavefront owns ROWS consecutive
// output rows x one 64-chunk (1 KiB) column segment.  The row index is wave-uniform, so the indices come through the
// scalar path (one s_load for all of the wavefront's rows, no vector load in front of the gather) and the
// wavefront's row loads are issued back to back before the first store.  Measured on 16 / 32 / 64 / 128 frames:
// one row per wavefront is best while the launch is a few rounds of wavefronts (more, shorter wavefronts drain
// evenly), two rows from about 64 k wavefronts on (+9 .. 15 %); four and eight rows are slower everywhere.
constexpr int kSplitWaves = 4;

template <typename IndexT, bool PAIR, int ROWS>
__global__ __launch_bounds__(64 * kSplitWaves) void split_wave_kernel(const uint4 *__restrict__ merged,
                                                                      const uint4 *__restrict__ merged_b,
                                                                      int64_t merged_rows,
                                                                      const IndexT *__restrict__ rev, int total,
                                                                      int chunks, uint4 *__restrict__ out,
                                                                      int segs, uint32_t n_waves, uint32_t run,
                                                                      uint32_t remapped_blocks, FastDiv by_run,
                                                                      FastDiv by_segs) {
    uint32_t bid = blockIdx.x;
    if (bid < remapped_blocks) {                            // runs of `run` workgroups stay on one XCD (one L2)
        const uint32_t local = bid >> 3;
        const uint32_t q = fast_div(local, by_run);
        bid = (q * 8u + (bid & 7u)) * run + (local - q * run);
    }
    const uint32_t wave = __builtin_amdgcn_readfirstlane(bid * kSplitWaves + (threadIdx.x >> 6));
    if (wave >= n_waves) return;
    const int lane = threadIdx.x & 63;
    const uint32_t group = fast_div(wave, by_segs);
    const int seg = static_cast<int>(wave - group * segs);
    const int row0 = static_cast<int>(group) * ROWS;
    const int out_chunks = PAIR ? 2 * chunks : chunks;
    const int out_chunk = seg * 64 + lane;
    const bool second = PAIR && seg * 64 >= chunks;          // wave-uniform: chunks is a multiple of 64
    const uint4 *__restrict__ src = second ? merged_b : merged;
    const int chunk = second ? out_chunk - chunks : out_chunk;
    uint4 *__restrict__ dst = out + static_cast<int64_t>(row0) * out_chunks + out_chunk;
    if (row0 + ROWS <= total) {
        // all indices first, then all row loads, then the stores: the wavefront's ROWS index -> row -> store
        // chains overlap instead of running one after the other
        int64_t s[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) s[r] = static_cast<int64_t>(rev[row0 + r]);
        uint4 v[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const bool ok = s[r] >= 0 && s[r] < merged_rows;
            v[r] = src[(ok ? s[r] : 0) * chunks + chunk];
            if (!ok) v[r] = make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < ROWS; ++r) st16_stream(dst + static_cast<int64_t>(r) * out_chunks, v[r]);
        return;
    }
    for (int r = 0; row0 + r < total; ++r) {                 // the last, partial group of rows
        const int64_t s = static_cast<int64_t>(rev[row0 + r]);
        uint4 v = make_uint4(0, 0, 0, 0);
        if (s >= 0 && s < merged_rows) v = src[s * chunks + chunk];
        st16_stream(dst + static_cast<int64_t>(r) * out_chunks, v);
    }
}

// The same for other widths of at least kFlatChunks chunks: a wavefront owns 128 consecutive chunks of the output, which
// lie in at most kFlatRows rows; their indices come through the scalar path, every lane takes its own.  Against a thread per
// chunk with an index load each, us, bf16, 768 channels: 96 frames of 1226 rows 54.5 -> 48.7, 128 71.6 -> 63.3 (6.0 TB/s), pairs
// of 128 148 -> 125; below 150 MB of output within 2 %.  Narrower rows lie too many to a wavefront: split_vec_kernel.
constexpr int kFlatRows = 4, kFlatChunks = 43;               // (127 / 43 + 2 rows)

template <typename IndexT, bool PAIR>
__global__ __launch_bounds__(64 * kSplitWaves) void split_flat_kernel(const uint4 *__restrict__ merged,
                                                                      const uint4 *__restrict__ merged_b, int64_t merged_rows,
                                                                      const IndexT *__restrict__ rev, int total, int chunks,
                                                                      uint4 *__restrict__ out, uint32_t items, uint32_t run,
                                                                      uint32_t remapped_blocks, FastDiv by_run, FastDiv by_out_chunks) {
    uint32_t bid = blockIdx.x;
    if (bid < remapped_blocks) {                            // runs of `run` workgroups stay on one XCD (one L2)
        const uint32_t local = bid >> 3;
        const uint32_t q = fast_div(local, by_run);
        bid = (q * 8u + (bid & 7u)) * run + (local - q * run);
    }
    const uint32_t first = __builtin_amdgcn_readfirstlane((bid * kSplitWaves + (threadIdx.x >> 6)) * 128u);
    if (first >= items) return;
    const int lane = threadIdx.x & 63;
    const int out_chunks = PAIR ? 2 * chunks : chunks;
    const int row0 = __builtin_amdgcn_readfirstlane(static_cast<int>(fast_div(first, by_out_chunks)));
    int64_t s[kFlatRows];
#pragma unroll
    for (int r = 0; r < kFlatRows; ++r) s[r] = static_cast<int64_t>(rev[min(row0 + r, total - 1)]);
    uint4 v[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const uint32_t id = min(first + 64u * u + lane, items - 1);
        const int row = static_cast<int>(fast_div(id, by_out_chunks)), out_chunk = static_cast<int>(id) - row * out_chunks;
        const bool second = PAIR && out_chunk >= chunks;
        const uint4 *__restrict__ src = second ? merged_b : merged;
        const int chunk = second ? out_chunk - chunks : out_chunk;
        int64_t from = s[0];
#pragma unroll
        for (int r = 1; r < kFlatRows; ++r) from = row - row0 == r ? s[r] : from;
        const bool ok = from >= 0 && from < merged_rows;
        v[u] = src[(ok ? from : 0) * chunks + chunk];
        if (!ok) v[u] = make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
        if (first + 64u * u + lane < items) st16_stream(out + first + 64u * u + lane, v[u]);
}

// element-wise fallback; `pair`: output rows are [row of merged | row of merged_b]
template <typename IndexT>
__global__ __launch_bounds__(kThreads) void split_elem_kernel(const uint8_t *__restrict__ merged,
                                                              const uint8_t *__restrict__ merged_b, bool pair,
                                                              int64_t merged_rows, const IndexT *__restrict__ rev,
                                                              int64_t total, int64_t row_bytes, int elem_bytes,
                                                              uint8_t *__restrict__ out) {
    const int64_t id = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    const int64_t per_row = row_bytes / elem_bytes;
    const int64_t per_out = pair ? 2 * per_row : per_row;
    if (id >= total * per_out) return;
    const int64_t i = id / per_out;
    const int64_t oc = id - i * per_out;
    const bool second = oc >= per_row;
    const uint8_t *__restrict__ src = second ? merged_b : merged;
    const int64_t c = second ? oc - per_row : oc;
    const int64_t s = static_cast<int64_t>(rev[i]);
    const bool ok = s >= 0 && s < merged_rows;
    if (elem_bytes == 4) {
        reinterpret_cast<uint32_t *>(out)[id] = ok ? reinterpret_cast<const uint32_t *>(src)[s * per_row + c] : 0u;
    } else {
        reinterpret_cast<uint16_t *>(out)[id] =
            ok ? reinterpret_cast<const uint16_t *>(src)[s * per_row + c] : uint16_t(0);
    }
}

template <int DT, bool DIRECT>
void launch_merge_vec(const MergeArgs &a, int64_t blocks, hipStream_t stream) {
    const MergeGeom &g = a.g;
    const dim3 grid(static_cast<unsigned>(blocks + (DIRECT ? 1 : 0))), block(kMergeThreads);
#define COME_MERGE_CASE(GH_, GW_)                                                              \
    if (g.gh == GH_ && g.gw == GW_) {                                                          \
        hipLaunchKernelGGL((merge_vec_kernel<DT, GH_, GW_, DIRECT>), grid, block, 0, stream, a);       \
        return;                                                                                \
    }
    COME_MERGE_CASE(3, 3)
    COME_MERGE_CASE(2, 2)
    COME_MERGE_CASE(1, 2)
    COME_MERGE_CASE(1, 4)
    COME_MERGE_CASE(1, 8)
    COME_MERGE_CASE(1, 9)
#undef COME_MERGE_CASE
    hipLaunchKernelGGL((merge_vec_kernel<DT, 0, 0, DIRECT>), grid, block, 0, stream, a);
}

template <int DT, int CH>
void launch_merge_narrow(const MergeArgs &a, bool direct, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(ceil_div(a.group_items, kThreads))), block(kThreads);
    if (direct) hipLaunchKernelGGL((merge_narrow_kernel<DT, CH, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((merge_narrow_kernel<DT, CH, false>), grid, block, 0, stream, a);
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace come

using namespace come;

static int merge_plan_impl(const char *who, const uint8_t *merge_mask, int64_t rows, int64_t groups, int64_t start_index,
                           int64_t group_size, int64_t tail, int32_t *offsets, int32_t *group_prefix, uint64_t *post,
                           uint32_t tag, void *stream) {
    COME_REQUIRE(rows >= 0 && groups >= 0, COME_ERR_INVALID, "%s: rows/groups must be >= 0", who);
    COME_REQUIRE(start_index >= 0, COME_ERR_INVALID, "%s: start_index must be >= 0", who);
    COME_REQUIRE(group_size > 0, COME_ERR_INVALID, "%s: group_size must be > 0", who);
    COME_REQUIRE(tail >= 0, COME_ERR_INVALID, "%s: tail must be >= 0", who);
    COME_REQUIRE(offsets != nullptr, COME_ERR_INVALID, "%s: offsets is NULL", who);
    COME_REQUIRE(rows * groups == 0 || (merge_mask && group_prefix), COME_ERR_INVALID,
                 "%s: merge_mask / group_prefix is NULL", who);
    const int64_t n_tok = start_index + groups * group_size + tail;
    COME_REQUIRE(rows < (1ll << 31) && groups < (1ll << 31) && rows * n_tok < (1ll << 31), COME_ERR_UNSUPPORTED,
                 "%s: rows * tokens per row must stay below 2^31", who);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (rows > 0 && aligned16(merge_mask) && rows * (rows - 1) / 2 <= kPlanRescanBytes / (groups > 0 ? groups : 1)) {
        hipLaunchKernelGGL(merge_plan_rows_kernel, dim3(static_cast<unsigned>(rows)), dim3(kPlanThreads), 0, s, merge_mask,
                           static_cast<int>(rows), static_cast<int>(groups), static_cast<int>(start_index),
                           static_cast<int>(group_size), static_cast<int>(tail), offsets, group_prefix, post, tag);
        COME_CHECK_LAUNCH(who);
        return COME_OK;
    }
    const int plan_groups = static_cast<int>(std::min<int64_t>(std::max<int64_t>((rows + kPlanRowsPerGroup - 1) / kPlanRowsPerGroup, 1), 2048));
    hipLaunchKernelGGL(merge_plan_kernel, dim3(plan_groups), dim3(64 * kPlanRowsPerGroup), 0, s, merge_mask,
                       static_cast<int>(rows), static_cast<int>(groups), static_cast<int>(start_index),
                       static_cast<int>(group_size), static_cast<int>(tail), offsets, group_prefix,
                       plan_groups > 1 ? nullptr : post, tag);
    if (plan_groups > 1)
        hipLaunchKernelGGL(merge_plan_scan_kernel, dim3(1), dim3(64), 0, s, offsets, static_cast<int>(rows), post, tag);
    COME_CHECK_LAUNCH(who);
    return COME_OK;
}

extern "C" int come_merge_plan(const uint8_t *merge_mask, int64_t rows, int64_t groups, int64_t start_index,
                               int64_t group_size, int64_t tail, int32_t *offsets, int32_t *group_prefix,
                               void *stream) {
    clear_error();
    return merge_plan_impl("come_merge_plan", merge_mask, rows, groups, start_index, group_size, tail, offsets,
                           group_prefix, nullptr, 0, stream);
}

extern "C" int come_merge_plan_post(const uint8_t *merge_mask, int64_t rows, int64_t groups, int64_t start_index,
                                    int64_t group_size, int64_t tail, int32_t *offsets, int32_t *group_prefix,
                                    uint64_t *post, uint32_t tag, void *stream) {
    clear_error();
    return merge_plan_impl("come_merge_plan_post", merge_mask, rows, groups, start_index, group_size, tail, offsets,
                           group_prefix, post, tag, stream);
}

static int token_merge_impl(const void *tokens, int dtype, int64_t rows, int64_t n_tok, int64_t chans, int64_t start_index,
                            int64_t group_h, int64_t group_w, int64_t grid_h, int64_t grid_w, const uint8_t *merge_mask,
                            const int32_t *offsets, const int32_t *group_prefix, void *out, int64_t out_rows,
                            int64_t *rev_i64, int32_t *rev_i32, float *weight_f32, int32_t *count_i32,
                            int64_t *offsets_i64, bool direct, uint64_t *post, uint32_t tag, void *stream) {
    COME_REQUIRE(dtype_ok(dtype), COME_ERR_UNSUPPORTED, "come_token_merge: unsupported dtype %d", dtype);
    COME_REQUIRE(rows >= 0 && n_tok >= 0 && chans >= 1 && out_rows >= 0, COME_ERR_INVALID,
                 "come_token_merge: negative size or chans < 1");
    COME_REQUIRE(start_index >= 0, COME_ERR_INVALID, "come_token_merge: start_index must be >= 0");
    COME_REQUIRE(group_h > 0 && group_w > 0, COME_ERR_INVALID, "come_token_merge: group_h and group_w must be > 0");
    COME_REQUIRE(grid_h >= 0 && grid_w >= 0, COME_ERR_INVALID, "come_token_merge: grid_h / grid_w must be >= 0");
    COME_REQUIRE(n_tok == start_index + grid_h * grid_w, COME_ERR_INVALID,
                 "come_token_merge: N != start_index + grid_h * grid_w (%lld != %lld + %lld * %lld)",
                 (long long)n_tok, (long long)start_index, (long long)grid_h, (long long)grid_w);
    COME_REQUIRE(rows * n_tok < (1ll << 31) && chans < (1ll << 24), COME_ERR_UNSUPPORTED,
                 "come_token_merge: rows * tokens per row must stay below 2^31");
    if (rows == 0 || n_tok == 0) return COME_OK;
    COME_REQUIRE(tokens && out && (offsets || direct), COME_ERR_INVALID, "come_token_merge: tokens / out / offsets is NULL");

    MergeArgs a{};
    MergeGeom &g = a.g;
    g.rows = static_cast<int>(rows);
    g.n_tok = static_cast<int>(n_tok);
    g.start = static_cast<int>(start_index);
    g.gh = static_cast<int>(group_h);
    g.gw = static_cast<int>(group_w);
    g.G = g.gh * g.gw;
    g.H = static_cast<int>(grid_h);
    g.W = static_cast<int>(grid_w);
    g.mw = g.W / g.gw;
    const int mh = g.H / g.gh;
    g.groups = mh * g.mw;
    g.cov_h = mh * g.gh;
    g.cov_w = g.mw * g.gw;
    g.tail = g.H * g.W - g.cov_h * g.cov_w;
    if (g.groups == 0) {            // no full window: every grid position is a leftover, row-major
        g.cov_h = 0;
        g.cov_w = 0;
        g.mw = 1;
    }
    g.out_rows = out_rows;
    COME_REQUIRE(g.groups == 0 || (merge_mask && (group_prefix || direct)), COME_ERR_INVALID,
                 "come_token_merge: merge_mask / group_prefix is NULL");
    a.post = post;
    a.post_tag = tag;
    a.tokens = tokens;
    a.out = out;
    a.mask = merge_mask;
    a.offsets = offsets;
    a.prefix = group_prefix;
    a.rev64 = rev_i64;
    a.rev32 = rev_i32;
    a.weight = weight_f32;
    a.count = count_i32;

    const int64_t row_bytes = chans * dtype_bytes(dtype);
    const bool vec = (row_bytes % 16 == 0) && aligned16(tokens) && aligned16(out);
    a.chunks = static_cast<int>(vec ? row_bytes / 16 : chans);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (chans <= kNarrowChans && !vec) {
        a.offsets64 = offsets_i64;
        a.group_items = rows * n_tok;
        a.by_groups = make_fastdiv(n_tok);
        a.by_per_row = make_fastdiv(g.W > 0 ? g.W : 1);
        a.by_chunks = make_fastdiv(g.gh);
        a.by_mw = make_fastdiv(g.gw);
#define COME_NARROW_CASE(CH_)                                                                                          \
    case CH_:                                                                                                          \
        if (dtype == COME_BF16) launch_merge_narrow<COME_BF16, CH_>(a, direct, s);                                     \
        else if (dtype == COME_F16) launch_merge_narrow<COME_F16, CH_>(a, direct, s);                                  \
        else launch_merge_narrow<COME_F32, CH_>(a, direct, s);                                                         \
        break;
        static_assert(kNarrowChans == 4, "one case per channel count");
        switch (chans) {
            COME_NARROW_CASE(1)
            COME_NARROW_CASE(2)
            COME_NARROW_CASE(3)
            COME_NARROW_CASE(4)
        }
#undef COME_NARROW_CASE
        COME_CHECK_LAUNCH("come_token_merge");
        return COME_OK;
    }
    const int threads = vec ? kMergeThreads : kThreads;
    a.by_chunks = make_fastdiv(a.chunks);
    a.by_groups = make_fastdiv(g.groups > 0 ? g.groups : 1);
    a.by_mw = make_fastdiv(g.mw > 0 ? g.mw : 1);
    a.by_per_row = make_fastdiv(g.start + g.tail > 0 ? g.start + g.tail : 1);
    a.by_side = make_fastdiv(g.W - g.cov_w > 0 ? g.W - g.cov_w : 1);
    // a launch of the 16-byte kernel covers fewer than 2^31 (unit, chunk) items of either kind; more rows take
    // several launches over consecutive row ranges (packed positions are absolute, so `out` stays where it is)
    const int64_t per_row_items = static_cast<int64_t>(g.groups > g.start + g.tail ? g.groups : g.start + g.tail) * a.chunks;
    int64_t rows_per_launch = rows;
    if (vec && per_row_items > 0) {
        rows_per_launch = ((1ll << 31) - 1) / per_row_items;
        COME_REQUIRE(rows_per_launch >= 1, COME_ERR_UNSUPPORTED,
                     "come_token_merge: more than 2^31 16-byte items in one row");
        if (rows_per_launch > rows) rows_per_launch = rows;
    }
    const int64_t tok_bytes = n_tok * row_bytes;
    for (int64_t f0 = 0; f0 < rows; f0 += rows_per_launch) {
        const int64_t nf = rows - f0 < rows_per_launch ? rows - f0 : rows_per_launch;
        g.rows = static_cast<int>(nf);
        a.tokens = static_cast<const char *>(tokens) + f0 * tok_bytes;
        a.mask = merge_mask ? merge_mask + f0 * g.groups : nullptr;
        a.offsets = direct ? nullptr : offsets + f0;
        a.offsets64 = offsets_i64 ? offsets_i64 + f0 : nullptr;
        a.prefix = group_prefix ? group_prefix + f0 * g.groups : nullptr;
        a.rev64 = rev_i64 ? rev_i64 + f0 * n_tok : nullptr;
        a.rev32 = rev_i32 ? rev_i32 + f0 * n_tok : nullptr;
        a.group_items = nf * g.groups * a.chunks;
        a.group_blocks = ceil_div(a.group_items, threads);
        a.single_items = nf * (g.start + g.tail) * a.chunks;
        const int64_t blocks = a.group_blocks + ceil_div(a.single_items, threads);
        COME_REQUIRE(blocks < (1ll << 31), COME_ERR_UNSUPPORTED, "come_token_merge: problem too large for one launch");
        if (blocks == 0) continue;
        if (vec) {
#define COME_VEC_CASE(DT_)                                            \
    if (direct) launch_merge_vec<DT_, true>(a, blocks, s);            \
    else launch_merge_vec<DT_, false>(a, blocks, s)
            if (dtype == COME_BF16) {
                COME_VEC_CASE(COME_BF16);
            } else if (dtype == COME_F16) {
                COME_VEC_CASE(COME_F16);
            } else {
                COME_VEC_CASE(COME_F32);
            }
#undef COME_VEC_CASE
        } else {
            const dim3 grid(static_cast<unsigned>(blocks)), block(kThreads);
            if (dtype == COME_BF16) hipLaunchKernelGGL(merge_elem_kernel<COME_BF16>, grid, block, 0, s, a);
            else if (dtype == COME_F16) hipLaunchKernelGGL(merge_elem_kernel<COME_F16>, grid, block, 0, s, a);
            else hipLaunchKernelGGL(merge_elem_kernel<COME_F32>, grid, block, 0, s, a);
        }
        COME_CHECK_LAUNCH("come_token_merge");
    }
    return COME_OK;
}

extern "C" int come_token_merge(const void *tokens, int dtype, int64_t rows, int64_t n_tok, int64_t chans,
                                int64_t start_index, int64_t group_h, int64_t group_w, int64_t grid_h,
                                int64_t grid_w, const uint8_t *merge_mask, const int32_t *offsets,
                                const int32_t *group_prefix, void *out, int64_t out_rows, int64_t *rev_i64,
                                int32_t *rev_i32, float *weight_f32, int32_t *count_i32, void *stream) {
    clear_error();
    return token_merge_impl(tokens, dtype, rows, n_tok, chans, start_index, group_h, group_w, grid_h, grid_w, merge_mask,
                            offsets, group_prefix, out, out_rows, rev_i64, rev_i32, weight_f32, count_i32, nullptr, false, nullptr, 0, stream);
}

extern "C" int come_token_merge_wide(const void *tokens, int dtype, int64_t rows, int64_t n_tok, int64_t chans,
                                     int64_t start_index, int64_t group_h, int64_t group_w, int64_t grid_h,
                                     int64_t grid_w, const uint8_t *merge_mask, const int32_t *offsets,
                                     const int32_t *group_prefix, void *out, int64_t out_rows, int64_t *rev_i64,
                                     int32_t *rev_i32, float *weight_f32, int32_t *count_i32, int64_t *offsets_i64,
                                     void *stream) {
    clear_error();
    return token_merge_impl(tokens, dtype, rows, n_tok, chans, start_index, group_h, group_w, grid_h, grid_w, merge_mask,
                            offsets, group_prefix, out, out_rows, rev_i64, rev_i32, weight_f32, count_i32, offsets_i64, false, nullptr, 0,
                            stream);
}

// What the DIRECT kernels take: a mask small enough to be counted by every wavefront (kDirectWindows), 16-byte aligned, rows of
// two 16-byte chunks or more, or of a few channels; one launch.
static bool direct_takes(const void *tokens, int dtype, int64_t rows, int64_t n_tok, int64_t chans, int64_t group_h, int64_t group_w,
                         int64_t grid_h, int64_t grid_w, const uint8_t *merge_mask) {
    if (!dtype_ok(dtype) || rows <= 0 || n_tok <= 0 || chans < 1 || chans >= (1ll << 24) || group_h <= 0 || group_w <= 0 || grid_h < group_h ||
        grid_w < group_w || rows >= (1ll << 31) || n_tok >= (1ll << 31) || rows * n_tok >= (1ll << 31))
        return false;
    const int64_t windows = rows * (grid_h / group_h) * (grid_w / group_w);
    if (windows > kDirectWindows || !aligned16(merge_mask)) return false;
    const int64_t row_bytes = chans * dtype_bytes(dtype);
    if (row_bytes % 16 == 0 && aligned16(tokens)) return row_bytes >= 32 && rows * n_tok * (row_bytes / 16) < (1ll << 31);
    return chans <= kNarrowChans;
}

// Where that saves time.  Above half of kDirectWindows a wavefront's share of the counting is up to 16 KB of mask, which only
// windows with enough of their own to move pay for (2 x 2 ones differ from run to run by what there is to gain); the plan of more than 2048 rows is slow (its scan is one wavefront's).  A
// call, merge behind its plan / direct, us, bf16: 16 384 windows of 1 x 2, 64 channels 10.7 / 11.5, 256 12.0 / 14.2, 1024 24.8 / 29.5;
// 2 x 2, 256 channels 15.2 / 15.6, 512 25.2 / 22.5 and 24.3 / 28.8, 1024 40.5 / 40.7 and 39.8 / 43.4; 3 x 3, 64 channels 12.1 / 12.5, 256 24.4 / 23.6, 1024 80.4 / 78.4;
// 12 288 windows of 3 x 3, 64 channels 11.8 / 12.3, 256 19.6 / 18.7; 8192 windows of 1 x 2, 64 channels 10.5 / 10.0, 1024 15.0 / 14.1;
// 3072 rows of 5 windows, 64 channels 36 / 11.8.
extern "C" int come_token_merge_is_direct(const void *tokens, int dtype, int64_t rows, int64_t n_tok, int64_t chans,
                                          int64_t group_h, int64_t group_w, int64_t grid_h, int64_t grid_w, const uint8_t *merge_mask) {
    if (!direct_takes(tokens, dtype, rows, n_tok, chans, group_h, group_w, grid_h, grid_w, merge_mask)) return 0;
    const int64_t windows = rows * (grid_h / group_h) * (grid_w / group_w), tokens_each = group_h * group_w;
    return windows <= kDirectWindows / 2 || rows > 2048 || chans <= kNarrowChans ||
           (tokens_each >= 8 && tokens_each * chans * dtype_bytes(dtype) >= 4096);
}

extern "C" int come_token_merge_direct(const void *tokens, int dtype, int64_t rows, int64_t n_tok, int64_t chans,
                                       int64_t start_index, int64_t group_h, int64_t group_w, int64_t grid_h,
                                       int64_t grid_w, const uint8_t *merge_mask, void *out, int64_t out_rows,
                                       int64_t *rev_i64, int32_t *rev_i32, float *weight_f32, int32_t *count_i32,
                                       int64_t *offsets_i64, uint64_t *post, uint32_t tag, void *stream) {
    clear_error();
    COME_REQUIRE(direct_takes(tokens, dtype, rows, n_tok, chans, group_h, group_w, grid_h, grid_w, merge_mask) &&
                     (chans * dtype_bytes(dtype) % 16 != 0 || aligned16(out)),
                 COME_ERR_UNSUPPORTED, "come_token_merge_direct: needs a plan (come_token_merge)");
    return token_merge_impl(tokens, dtype, rows, n_tok, chans, start_index, group_h, group_w, grid_h, grid_w, merge_mask, nullptr,
                            nullptr, out, out_rows, rev_i64, rev_i32, weight_f32, count_i32, offsets_i64, true, post, tag, stream);
}

// shared body of come_token_split (pair = false, merged_b unused) and come_token_split_pair
static int token_split_impl(const char *who, bool pair, const void *merged, const void *merged_b, int dtype,
                            int64_t merged_rows, int64_t chans, const int64_t *rev_i64, const int32_t *rev_i32,
                            int64_t total, void *out, void *stream) {
    COME_REQUIRE(dtype_ok(dtype), COME_ERR_UNSUPPORTED, "%s: unsupported dtype %d", who, dtype);
    COME_REQUIRE(merged_rows >= 0 && chans >= 1 && total >= 0, COME_ERR_INVALID,
                 "%s: negative size or chans < 1", who);
    COME_REQUIRE((rev_i64 != nullptr) != (rev_i32 != nullptr) || total == 0, COME_ERR_INVALID,
                 "%s: exactly one of rev_i64 / rev_i32 must be given", who);
    if (total == 0) return COME_OK;
    COME_REQUIRE(out != nullptr && (merged_rows == 0 || (merged != nullptr && (!pair || merged_b != nullptr))),
                 COME_ERR_INVALID, "%s: merged / out is NULL", who);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t row_bytes = chans * dtype_bytes(dtype);
    const bool vec = (row_bytes % 16 == 0) && aligned16(merged) && aligned16(merged_b) && aligned16(out);
    if (vec) {
        const int chunks = static_cast<int>(row_bytes / 16);
        const int out_chunks = pair ? 2 * chunks : chunks;
        COME_REQUIRE(out_chunks < (1 << 23), COME_ERR_UNSUPPORTED, "%s: rows wider than 128 MiB are not supported", who);
        const FastDiv by_out_chunks = make_fastdiv(out_chunks);
        // a launch covers fewer than 2^31 (row, 16-byte chunk) items; larger outputs take several launches over
        // consecutive row ranges (whole XCD runs each)
        int64_t rows_per_launch = ((1ll << 31) - 1) / out_chunks;
        if (rows_per_launch > kSplitRunRows) rows_per_launch -= rows_per_launch % kSplitRunRows;
        const int run_rows = (merged_rows + total) * row_bytes * (pair ? 2 : 1) > kSplitLarge ? kSplitRunRowsLarge : kSplitRunRows;
        for (int64_t r0 = 0; r0 < total; r0 += rows_per_launch) {
            const int64_t nr = total - r0 < rows_per_launch ? total - r0 : rows_per_launch;
            const int64_t items = nr * out_chunks;
            if (out_chunks % 64 == 0 && chunks % 64 == 0 && merged_rows > 0) {
                const int segs = out_chunks / 64;
                const int wave_rows = nr * segs > 65536 ? 2 : 1;
                const int64_t n_waves = ceil_div(nr, wave_rows) * segs;
                const int64_t wrun64 = static_cast<int64_t>(run_rows) / wave_rows * segs / kSplitWaves;
                const uint32_t wrun = static_cast<uint32_t>(wrun64 < 1 ? 1 : wrun64);
                const dim3 wgrid(static_cast<unsigned>(ceil_div(n_waves, kSplitWaves))), wblock(64 * kSplitWaves);
                const uint4 *a4 = static_cast<const uint4 *>(merged), *b4 = static_cast<const uint4 *>(merged_b);
                uint4 *o4 = static_cast<uint4 *>(out) + r0 * out_chunks;
#define COME_SPLITW_ROWS(IDX_, PAIR_, REV_, ROWS_)                                                                  \
    hipLaunchKernelGGL((split_wave_kernel<IDX_, PAIR_, ROWS_>), wgrid, wblock, 0, s, a4, b4, merged_rows,           \
                       REV_ + r0, static_cast<int>(nr), chunks, o4, segs, static_cast<uint32_t>(n_waves), wrun,     \
                       (wgrid.x / (8u * wrun)) * (8u * wrun), make_fastdiv(wrun), make_fastdiv(segs))
#define COME_SPLITW_CASE(IDX_, PAIR_, REV_)                                 \
    do {                                                                    \
        if (wave_rows == 2) COME_SPLITW_ROWS(IDX_, PAIR_, REV_, 2);         \
        else COME_SPLITW_ROWS(IDX_, PAIR_, REV_, 1);                        \
    } while (0)
                if (rev_i64 && pair) COME_SPLITW_CASE(int64_t, true, rev_i64);
                else if (rev_i64) COME_SPLITW_CASE(int64_t, false, rev_i64);
                else if (pair) COME_SPLITW_CASE(int32_t, true, rev_i32);
                else COME_SPLITW_CASE(int32_t, false, rev_i32);
#undef COME_SPLITW_CASE
#undef COME_SPLITW_ROWS
                COME_CHECK_LAUNCH(who);
                continue;
            }
            if (out_chunks >= kFlatChunks && merged_rows > 0) {
                const uint32_t blocks = static_cast<uint32_t>(ceil_div(items, 128 * kSplitWaves));
                const int64_t frun64 = static_cast<int64_t>(run_rows) * out_chunks / (128 * kSplitWaves);
                const uint32_t frun = static_cast<uint32_t>(frun64 < 1 ? 1 : frun64);
                const uint4 *a4 = static_cast<const uint4 *>(merged), *b4 = static_cast<const uint4 *>(merged_b);
                uint4 *o4 = static_cast<uint4 *>(out) + r0 * out_chunks;
#define COME_FLAT_CASE(IDX_, PAIR_, REV_)                                                                                        \
    hipLaunchKernelGGL((split_flat_kernel<IDX_, PAIR_>), dim3(blocks), dim3(64 * kSplitWaves), 0, s, a4, b4, merged_rows,       \
                       REV_ + r0, static_cast<int>(nr), chunks, o4, static_cast<uint32_t>(items), frun,                         \
                       (blocks / (8u * frun)) * (8u * frun), make_fastdiv(frun), by_out_chunks)
                if (rev_i64 && pair) COME_FLAT_CASE(int64_t, true, rev_i64);
                else if (rev_i64) COME_FLAT_CASE(int64_t, false, rev_i64);
                else if (pair) COME_FLAT_CASE(int32_t, true, rev_i32);
                else COME_FLAT_CASE(int32_t, false, rev_i32);
#undef COME_FLAT_CASE
                COME_CHECK_LAUNCH(who);
                continue;
            }
            const int64_t run64 = static_cast<int64_t>(run_rows) * out_chunks / kThreads;
            const uint32_t run = static_cast<uint32_t>(run64 < 1 ? 1 : run64);
            const dim3 grid(static_cast<unsigned>(ceil_div(items, kThreads))), block(kThreads);
            const uint4 *a4 = static_cast<const uint4 *>(merged), *b4 = static_cast<const uint4 *>(merged_b);
            uint4 *o4 = static_cast<uint4 *>(out) + r0 * out_chunks;
#define COME_SPLIT_CASE(IDX_, PAIR_, REV_)                                                                       \
    hipLaunchKernelGGL((split_vec_kernel<IDX_, PAIR_>), grid, block, 0, s, a4, b4, merged_rows, REV_ + r0,       \
                       chunks, o4, items, by_out_chunks, run)
            if (rev_i64 && pair) COME_SPLIT_CASE(int64_t, true, rev_i64);
            else if (rev_i64) COME_SPLIT_CASE(int64_t, false, rev_i64);
            else if (pair) COME_SPLIT_CASE(int32_t, true, rev_i32);
            else COME_SPLIT_CASE(int32_t, false, rev_i32);
            COME_CHECK_LAUNCH(who);
        }
#undef COME_SPLIT_CASE
    } else {
        const int eb = dtype_bytes(dtype);
        const int64_t blocks = ceil_div(total * chans * (pair ? 2 : 1), kThreads);
        COME_REQUIRE(blocks < (1ll << 31), COME_ERR_UNSUPPORTED, "%s: problem too large for one launch", who);
        const dim3 grid(static_cast<unsigned>(blocks)), block(kThreads);
        const uint8_t *a1 = static_cast<const uint8_t *>(merged), *b1 = static_cast<const uint8_t *>(merged_b);
        if (rev_i64)
            hipLaunchKernelGGL(split_elem_kernel<int64_t>, grid, block, 0, s, a1, b1, pair, merged_rows, rev_i64, total,
                               row_bytes, eb, static_cast<uint8_t *>(out));
        else
            hipLaunchKernelGGL(split_elem_kernel<int32_t>, grid, block, 0, s, a1, b1, pair, merged_rows, rev_i32, total,
                               row_bytes, eb, static_cast<uint8_t *>(out));
    }
    COME_CHECK_LAUNCH(who);
    return COME_OK;
}

extern "C" int come_token_split(const void *merged, int dtype, int64_t merged_rows, int64_t chans,
                                const int64_t *rev_i64, const int32_t *rev_i32, int64_t total, void *out,
                                void *stream) {
    clear_error();
    return token_split_impl("come_token_split", false, merged, nullptr, dtype, merged_rows, chans, rev_i64, rev_i32, total,
                            out, stream);
}

extern "C" int come_token_split_pair(const void *merged_a, const void *merged_b, int dtype, int64_t merged_rows,
                                     int64_t chans, const int64_t *rev_i64, const int32_t *rev_i32, int64_t total,
                                     void *out, void *stream) {
    clear_error();
    return token_split_impl("come_token_split_pair", true, merged_a, merged_b, dtype, merged_rows, chans, rev_i64, rev_i32,
                            total, out, stream);
}
