// Suffix operators on packed segments: append T dense rows to every segment, or strip them again.
// Both are row copies (HBM-bound byte work).  Small tensors, and rows that are no multiple of 16 bytes: one thread per
// (output row, 16-byte chunk or element) finds its segment by bisection over the segment offsets and copies from the packed
// rows or from the dense suffix block.  Large tensors of 16-byte chunks: a wavefront owns 256 consecutive chunks of the
// output, finds the segment of the first by a scalar bisection and, where all of them come from that segment's body (a copy
// at a fixed distance), moves four per lane back to back.
#include "come_common.h"

namespace come {
namespace {

constexpr int kThreads = 256;

struct SuffixArgs {
    const uint8_t *tokens;        // [rows_in, row_bytes]
    const float *weight;          // [rows_in] or nullptr
    const int64_t *offsets;       // [n_seg + 1] boundaries of the input segments
    const uint8_t *suffix_in;     // add: [n_seg, T, row_bytes]
    uint8_t *out_tokens;          // add: [rows_in + n_seg T, ..]; strip: [rows_in - n_seg T, ..]
    float *out_weight;
    int64_t *out_offsets;         // [n_seg + 1]
    uint8_t *suffix_out;          // strip: [n_seg, T, row_bytes]
    int64_t rows_in, rows_out, n_seg, T;
    int64_t row_bytes;
    int unit;                     // bytes moved per thread: 16, 4 or 2
    int units_per_row;
    int strip;                    // 0 = append, 1 = strip
    FastDiv by_units;             // 16-byte kernel: units_per_row
    uint64_t *post;               // strip, optional: host memory that receives 1 if some segment is shorter than T, else 0
    uint32_t post_tag;
};

// largest s in [lo, hi] with start(s) <= row, where start(s) = offsets[s] + s * step
__device__ inline int64_t find_segment(const int64_t *offsets, int64_t lo, int64_t hi, int64_t step, int64_t row) {
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) >> 1;
        if (offsets[mid] + mid * step <= row) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__device__ inline void copy_unit(uint8_t *dst, const uint8_t *src, int unit) {
    if (unit == 16) *reinterpret_cast<uint4 *>(dst) = *reinterpret_cast<const uint4 *>(src);
    else if (unit == 4) *reinterpret_cast<uint32_t *>(dst) = *reinterpret_cast<const uint32_t *>(src);
    else *reinterpret_cast<uint16_t *>(dst) = *reinterpret_cast<const uint16_t *>(src);
}

// What the host waits for (whether some segment is shorter than T) and the new boundaries.
__device__ inline void verdict_and_offsets(const SuffixArgs &a) {
    if (a.post != nullptr && blockIdx.x == 0) {                          // first thing the launch does
        __shared__ int too_short;
        if (threadIdx.x == 0) too_short = 0;
        __syncthreads();
        for (int64_t s = threadIdx.x; s < a.n_seg; s += kThreads)
            if (a.offsets[s + 1] - a.offsets[s] < a.T) too_short = 1;
        __syncthreads();
        if (threadIdx.x == 0) post_to_host(a.post, a.post_tag, static_cast<uint32_t>(too_short));
    }
    for (int64_t id = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; id <= a.n_seg && a.out_offsets != nullptr;
         id += static_cast<int64_t>(gridDim.x) * kThreads)               // n_seg + 1 of them
        a.out_offsets[id] = a.offsets[id] + (a.strip ? -id : id) * a.T;
}

// Where an output row (of the body, or behind it of the returned suffix block) comes from, and where it goes to;
// its segment is known to lie in [lo, hi].
struct Move {
    const uint8_t *src;
    uint8_t *dst;
    int64_t weight_row;            // input row whose weight goes with it, -1: none
};
__device__ inline Move locate_row(const SuffixArgs &a, int64_t row, int64_t lo, int64_t hi) {
    if (row < a.rows_out) {
        const int64_t step = a.strip ? -a.T : a.T;
        const int64_t s = find_segment(a.offsets, lo, hi, step, row);
        const int64_t j = row - (a.offsets[s] + s * step);               // position inside the output segment
        const int64_t len_in = a.offsets[s + 1] - a.offsets[s];
        // The offsets come from device memory that the host cannot check: indices derived from them are clamped
        // into the tensors, so that inconsistent offsets give wrong rows instead of accesses outside them.
        uint8_t *const dst = a.out_tokens + row * a.row_bytes;
        if (a.rows_in > 0 && (a.strip || j < len_in || a.T == 0)) {
            const int64_t r = min(max(a.offsets[s] + j, int64_t{0}), a.rows_in - 1);
            return {a.tokens + r * a.row_bytes, dst, r};
        }
        const int64_t t = min(max(j - len_in, int64_t{0}), a.T - 1);
        return {a.suffix_in + (s * a.T + t) * a.row_bytes, dst, -1};
    }
    const int64_t e = row - a.rows_out;                                  // (segment, t) of the stripped block
    const int64_t s = e / a.T;
    const int64_t t = e - s * a.T;
    // a segment shorter than T (caller error) or inconsistent offsets stay in bounds
    const int64_t r = min(max(a.offsets[s + 1] - a.T + t, int64_t{0}), a.rows_in - 1);
    return {a.tokens + r * a.row_bytes, a.suffix_out + e * a.row_bytes, -1};
}
__device__ inline float weight_of(const SuffixArgs &a, const Move &m) {
    return a.weight != nullptr && m.weight_row >= 0 ? a.weight[m.weight_row] : 1.f;
}

__global__ __launch_bounds__(kThreads) void suffix_kernel(const SuffixArgs a) {
    verdict_and_offsets(a);
    const int64_t id = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    const int64_t row = id / a.units_per_row;
    if (row >= a.rows_out + (a.strip ? a.n_seg * a.T : 0)) return;
    const int64_t col = (id - row * a.units_per_row) * a.unit;
    const Move m = locate_row(a, row, 0, a.n_seg - 1);
    const float w = weight_of(a, m);                                     // (on its way beside the copy, not behind it)
    copy_unit(m.dst + col, m.src + col, a.unit);
    if (col == 0 && row < a.rows_out && a.out_weight) a.out_weight[row] = w;
}

// The 16-byte form for large tensors.  A thread per chunk (the kernel above) puts a 64-bit division and two dependent loads
// of the offsets in front of every thread's one load; here they are scalar and made once for 256 chunks, and a lane has four
// loads in flight.  Two segments of 51 200 and 38 400 rows of 1024 bf16, two rows appended and stripped again: 142 -> 118 us
// (5.2 -> 6.2 TB/s; half of that size 64.9 -> 57.1 us).
// Streaming accesses keep what a launch moves out of the 256 MiB last-level cache.  They pay where it could not stay there
// anyhow: 367 MB moved by each of the two launches 129 us cached, 118 streamed; 275 MB 85.9 and 89.2 (the second launch
// still finds what the first one wrote).  A small launch is latency, and the smaller kernel's is 1 us shorter: below 20 MiB
// of output it stays in use (1400 rows of 384 bf16: 16.4 us there, 17.9 here; 17 MB 20.9 and 21.6; 23 MB 22.6 and 21.5).
constexpr int kCopies = 4;                                               // chunks per lane
constexpr int64_t kRowsChunks = 5ll << 18;
constexpr int64_t kStreamBytes = 320ll << 20;

template <bool STREAM>
__global__ __launch_bounds__(kThreads) void suffix_rows_kernel(const SuffixArgs a, const int64_t *__restrict__ offsets) {
    verdict_and_offsets(a);
    const uint32_t units = static_cast<uint32_t>(a.units_per_row);
    const uint32_t items = static_cast<uint32_t>((a.rows_out + (a.strip ? a.n_seg * a.T : 0)) * units);      // < 2^31
    const uint32_t first = __builtin_amdgcn_readfirstlane((blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6)) * (64u * kCopies));
    if (first >= items) return;
    const uint32_t lane = threadIdx.x & 63, last = min(first + 64u * kCopies, items) - 1;
    const uint32_t row0 = __builtin_amdgcn_readfirstlane(fast_div(first, a.by_units));
    const uint32_t row1 = __builtin_amdgcn_readfirstlane(fast_div(last, a.by_units));
    const int64_t step = a.strip ? -a.T : a.T;
    const int64_t s0 = find_segment(offsets, 0, a.n_seg - 1, step, row0);
    const int64_t back = s0 * step;                                      // input row = output row - back
    const int64_t start = offsets[s0] + back, end = offsets[s0 + 1] + back - (a.strip ? a.T : 0);   // the segment's body
    uint4 v[kCopies];
    if (row0 >= start && row1 < min(end, a.rows_out) && row0 - back >= 0 && row1 - back < a.rows_in) {
        const uint4 *const src = reinterpret_cast<const uint4 *>(a.tokens) - back * static_cast<int64_t>(units);
        uint4 *const dst = reinterpret_cast<uint4 *>(a.out_tokens);
#pragma unroll
        for (int u = 0; u < kCopies; ++u) {
            const uint4 *const p = src + min(first + 64u * u + lane, last);
            v[u] = STREAM ? ld16_stream(p) : *p;
        }
        if (a.out_weight != nullptr)                                     // the rows whose first chunk lies in these
            for (uint32_t r = row0 + (row0 * units != first) + lane; r <= row1; r += 64)
                a.out_weight[r] = a.weight != nullptr ? a.weight[r - back] : 1.f;
#pragma unroll
        for (int u = 0; u < kCopies; ++u) {
            const uint32_t id = first + 64u * u + lane;
            if (id <= last) {
                if (STREAM) st16_stream(dst + id, v[u]);
                else dst[id] = v[u];
            }
        }
        return;
    }
    const int64_t s1 = row1 >= a.rows_out ? a.n_seg - 1 : find_segment(offsets, s0, a.n_seg - 1, step, row1);
    uint4 *to[kCopies];
    float w[kCopies];
    int64_t weight_to[kCopies];
#pragma unroll
    for (int u = 0; u < kCopies; ++u) {
        const uint32_t id = min(first + 64u * u + lane, last);
        const uint32_t row = fast_div(id, a.by_units), col = id - row * units;
        const Move m = locate_row(a, row, s0, s1);
        v[u] = reinterpret_cast<const uint4 *>(m.src)[col];
        to[u] = reinterpret_cast<uint4 *>(m.dst) + col;
        w[u] = weight_of(a, m);
        weight_to[u] = col == 0 && row < a.rows_out && a.out_weight != nullptr ? static_cast<int64_t>(row) : -1;
    }
#pragma unroll
    for (int u = 0; u < kCopies; ++u) {
        if (first + 64u * u + lane <= last) *to[u] = v[u];
        if (weight_to[u] >= 0) a.out_weight[weight_to[u]] = w[u];
    }
}

int launch(SuffixArgs &a, int dtype, int64_t chans, const void *const *ptrs, int n_ptrs, void *stream, const char *what) {
    a.row_bytes = chans * dtype_bytes(dtype);
    bool aligned = a.row_bytes % 16 == 0;
    for (int i = 0; i < n_ptrs; ++i) aligned = aligned && (reinterpret_cast<uintptr_t>(ptrs[i]) & 15u) == 0;
    a.unit = aligned ? 16 : dtype_bytes(dtype);
    a.units_per_row = static_cast<int>(a.row_bytes / a.unit);
    const int64_t rows = a.rows_out + (a.strip ? a.n_seg * a.T : 0);
    int64_t items = rows * a.units_per_row;
    if (items < 1) items = 1;                                            // the offsets are written in any case
    if (aligned && items >= kRowsChunks && items < (1ll << 31)) {
        a.by_units = make_fastdiv(a.units_per_row);
        const bool stream_it = 32 * items > kStreamBytes;                // read and written
        hipLaunchKernelGGL(stream_it ? suffix_rows_kernel<true> : suffix_rows_kernel<false>,
                           dim3(static_cast<unsigned>(ceil_div(items, kThreads * kCopies))), dim3(kThreads), 0,
                           static_cast<hipStream_t>(stream), a, a.offsets);
        COME_CHECK_LAUNCH(what);
        return COME_OK;
    }
    const int64_t blocks = ceil_div(items, kThreads);
    COME_REQUIRE(blocks < (1ll << 31), COME_ERR_UNSUPPORTED, "%s: problem too large for one launch", what);
    hipLaunchKernelGGL(suffix_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0,
                       static_cast<hipStream_t>(stream), a);
    COME_CHECK_LAUNCH(what);
    return COME_OK;
}

}  // namespace
}  // namespace come

using namespace come;

extern "C" int come_jagged_add_suffix(const void *tokens, const float *weight, int dtype, int64_t rows, int64_t chans,
                                      const int64_t *offsets, int64_t n_seg, const void *suffix, int64_t count,
                                      void *out_tokens, float *out_weight, int64_t *out_offsets, void *stream) {
    clear_error();
    COME_REQUIRE(dtype_ok(dtype), COME_ERR_UNSUPPORTED, "come_jagged_add_suffix: unsupported dtype %d", dtype);
    COME_REQUIRE(rows >= 0 && chans >= 1 && n_seg >= 0 && count >= 0, COME_ERR_INVALID,
                 "come_jagged_add_suffix: negative size or chans < 1");
    COME_REQUIRE(chans < (1ll << 24) && n_seg < (1ll << 31), COME_ERR_UNSUPPORTED, "come_jagged_add_suffix: too large");
    COME_REQUIRE(offsets && out_offsets, COME_ERR_INVALID, "come_jagged_add_suffix: offsets is NULL");
    COME_REQUIRE(n_seg > 0 || rows == 0, COME_ERR_INVALID, "come_jagged_add_suffix: rows without segments");
    COME_REQUIRE((rows == 0 || tokens) && (n_seg * count == 0 || suffix) && (rows + n_seg * count == 0 || out_tokens),
                 COME_ERR_INVALID, "come_jagged_add_suffix: NULL tensor");
    COME_REQUIRE((weight == nullptr) == (out_weight == nullptr) || rows == 0, COME_ERR_INVALID,
                 "come_jagged_add_suffix: weight and out_weight go together");
    SuffixArgs a{};
    a.tokens = static_cast<const uint8_t *>(tokens);
    a.weight = weight;
    a.offsets = offsets;
    a.suffix_in = static_cast<const uint8_t *>(suffix);
    a.out_tokens = static_cast<uint8_t *>(out_tokens);
    a.out_weight = out_weight;
    a.out_offsets = out_offsets;
    a.rows_in = rows;
    a.rows_out = rows + n_seg * count;
    a.n_seg = n_seg;
    a.T = count;
    a.strip = 0;
    const void *ptrs[3] = {tokens, suffix, out_tokens};
    return launch(a, dtype, chans, ptrs, 3, stream, "come_jagged_add_suffix");
}

static int split_suffix_impl(const void *tokens, const float *weight, int dtype, int64_t rows, int64_t chans,
                             const int64_t *offsets, int64_t n_seg, int64_t count, void *out_tokens, float *out_weight,
                             int64_t *out_offsets, void *out_suffix, uint64_t *post, uint32_t tag, void *stream) {
    COME_REQUIRE(dtype_ok(dtype), COME_ERR_UNSUPPORTED, "come_jagged_split_suffix: unsupported dtype %d", dtype);
    COME_REQUIRE(rows >= 0 && chans >= 1 && n_seg >= 0 && count >= 0, COME_ERR_INVALID,
                 "come_jagged_split_suffix: negative size or chans < 1");
    COME_REQUIRE(chans < (1ll << 24) && n_seg < (1ll << 31), COME_ERR_UNSUPPORTED, "come_jagged_split_suffix: too large");
    COME_REQUIRE(rows - n_seg * count >= 0, COME_ERR_INVALID,
                 "come_jagged_split_suffix: cannot strip %lld rows from each of %lld segments (%lld rows in total)",
                 (long long)count, (long long)n_seg, (long long)rows);
    COME_REQUIRE(offsets && out_offsets, COME_ERR_INVALID, "come_jagged_split_suffix: offsets is NULL");
    COME_REQUIRE(n_seg > 0 || rows == 0, COME_ERR_INVALID, "come_jagged_split_suffix: rows without segments");
    COME_REQUIRE((rows == 0 || tokens) && (rows - n_seg * count == 0 || out_tokens) && (n_seg * count == 0 || out_suffix),
                 COME_ERR_INVALID, "come_jagged_split_suffix: NULL tensor");
    COME_REQUIRE((weight == nullptr) == (out_weight == nullptr) || rows - n_seg * count == 0, COME_ERR_INVALID,
                 "come_jagged_split_suffix: weight and out_weight go together");
    SuffixArgs a{};
    a.tokens = static_cast<const uint8_t *>(tokens);
    a.weight = weight;
    a.offsets = offsets;
    a.out_tokens = static_cast<uint8_t *>(out_tokens);
    a.out_weight = out_weight;
    a.out_offsets = out_offsets;
    a.suffix_out = static_cast<uint8_t *>(out_suffix);
    a.rows_in = rows;
    a.rows_out = rows - n_seg * count;
    a.n_seg = n_seg;
    a.T = count;
    a.strip = 1;
    a.post = post;
    a.post_tag = tag;
    const void *ptrs[3] = {tokens, out_tokens, out_suffix};
    return launch(a, dtype, chans, ptrs, 3, stream, "come_jagged_split_suffix");
}

extern "C" int come_jagged_split_suffix(const void *tokens, const float *weight, int dtype, int64_t rows,
                                        int64_t chans, const int64_t *offsets, int64_t n_seg, int64_t count,
                                        void *out_tokens, float *out_weight, int64_t *out_offsets, void *out_suffix,
                                        void *stream) {
    clear_error();
    return split_suffix_impl(tokens, weight, dtype, rows, chans, offsets, n_seg, count, out_tokens, out_weight, out_offsets,
                             out_suffix, nullptr, 0, stream);
}

extern "C" int come_jagged_split_suffix_post(const void *tokens, const float *weight, int dtype, int64_t rows,
                                             int64_t chans, const int64_t *offsets, int64_t n_seg, int64_t count,
                                             void *out_tokens, float *out_weight, int64_t *out_offsets,
                                             void *out_suffix, uint64_t *post, uint32_t tag, void *stream) {
    clear_error();
    return split_suffix_impl(tokens, weight, dtype, rows, chans, offsets, n_seg, count, out_tokens, out_weight, out_offsets,
                             out_suffix, post, tag, stream);
}
