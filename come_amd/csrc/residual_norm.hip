// What stands between two linear layers of a pre-norm transformer block: x + scale * y (LayerScale and residual) and the
// LayerNorm of the sum, in one pass over memory.  Also the LayerNorm alone, of rows that lie in equally spaced groups (the
// patch tokens of every frame behind its special tokens).
//
// HBM-bound: two rows read, two written.  As separate tensor operations (product, sum, LayerNorm) the same step reads four
// rows and writes three.  A wavefront owns a row: its 16-byte chunks stay in registers (K of them per lane) through both
// passes of the statistics, the sums run over lanes by data-parallel-primitive moves, nothing goes through LDS.  Four
// wavefronts a workgroup; all of a row's loads are in flight before the first is looked at.
// 25 536 rows of 1024 bf16: 95 us as separate operations, 36.5 us here (209 MB, 5.7 TB/s).  LayerNorm of 32 x 1369 rows of
// 2048 behind 5 special tokens each: copy and LayerNorm 204 us, 62 us here (359 MB, 5.8 TB/s).
//
// Rounding: that of the separate operations.  The product is rounded to the storage dtype, the sum is rounded, and the
// normalised value is taken from the rounded sum; mean and variance (two passes, in registers) are fp32.
#include "come_common.h"

namespace come {
namespace {

struct ResidualArgs {
    const char *x, *y;               // y: nullptr = no residual step
    const float *partial;            // SPLITS > 0: y as so many fp32 sums, [SPLITS][rows][C] ...
    const char *y_bias;              // ... and what is added to them, [C] or nullptr
    const char *scale;               // [C]
    const char *weight, *bias;       // [C] or nullptr
    char *sum_out, *norm_out;        // either may be nullptr
    int64_t rows;
    int64_t group_rows;              // consecutive rows of x that lie one behind another
    int64_t group_bytes;             // from one such group to the next
    int64_t row_bytes;
    int chunks;                      // 16-byte chunks a row
    float inv_c, eps;
};

// Sum over the wavefront, the same in every lane (a fixed order of additions).
__device__ inline float wave_sum(float v) {
    auto step = [&](float t) { v += t; };
    step(__uint_as_float(dpp_take<kRowShr1, 0xf>(0u, __float_as_uint(v))));
    step(__uint_as_float(dpp_take<kRowShr2, 0xf>(0u, __float_as_uint(v))));
    step(__uint_as_float(dpp_take<kRowShr4, 0xf>(0u, __float_as_uint(v))));
    step(__uint_as_float(dpp_take<kRowShr8, 0xf>(0u, __float_as_uint(v))));
    step(__uint_as_float(dpp_take<kRowBcast15, 0xa>(0u, __float_as_uint(v))));
    step(__uint_as_float(dpp_take<kRowBcast31, 0xc>(0u, __float_as_uint(v))));
    return __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(__float_as_uint(v)), 63)));
}

// K: chunks per lane.  Chunk c of a row belongs to lane c % 64.  SPLITS: y comes as sums over shares of the product behind it
// (come_linear_split), which meet here, get their bias and are rounded as the product's own result would be.
template <int DT, int K, int SPLITS>
__global__ void __launch_bounds__(256) residual_norm_kernel(const ResidualArgs a) {
#pragma clang fp contract(off)               // (the product is rounded before it is added, in fp32 as well)
    using V = Vec16<DT>;
    const int lane = threadIdx.x & 63;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    if (row >= a.rows) return;
    const int64_t at = row * a.row_bytes;
    const char *const x = a.group_rows >= a.rows ? a.x + at : a.x + row / a.group_rows * a.group_bytes + row % a.group_rows * a.row_bytes;
    uint4 xr[K], yr[K], sc[K], wr[K], br[K];          // (gain and shift of the norm: short launches would wait for them at the end)
    bool live[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        live[k] = lane + 64 * k < a.chunks;
        xr[k] = yr[k] = sc[k] = wr[k] = br[k] = make_uint4(0, 0, 0, 0);
        if (live[k]) {
            const int c = (lane + 64 * k) * 16;
            if (a.norm_out != nullptr && a.weight != nullptr) wr[k] = ld16(reinterpret_cast<const uint4 *>(a.weight + c));
            if (a.norm_out != nullptr && a.bias != nullptr) br[k] = ld16(reinterpret_cast<const uint4 *>(a.bias + c));
            xr[k] = ld16(reinterpret_cast<const uint4 *>(x + c));
            if (SPLITS > 0 || a.y != nullptr) {
                if (SPLITS == 0) yr[k] = ld16(reinterpret_cast<const uint4 *>(a.y + at + c));
                sc[k] = ld16(reinterpret_cast<const uint4 *>(a.scale + c));
            }
        }
    }
    if constexpr (SPLITS > 0) {
        static_assert(V::N == 8, "16-bit types");
        float4 part[K][SPLITS][2];
        uint4 bias[K];
        const int64_t row_floats = a.row_bytes / 2;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            bias[k] = make_uint4(0, 0, 0, 0);
            if (live[k] && a.y_bias != nullptr) bias[k] = ld16(reinterpret_cast<const uint4 *>(a.y_bias + (lane + 64 * k) * 16));
#pragma unroll
            for (int s = 0; s < SPLITS; ++s)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    part[k][s][i] = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (live[k])
                        part[k][s][i] = *reinterpret_cast<const float4 *>(a.partial + (s * a.rows + row) * row_floats + (lane + 64 * k) * 8 + 4 * i);
                }
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            float f[V::N];
            V::unpack(bias[k], f);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                float4 sum = part[k][0][i];
#pragma unroll
                for (int s = 1; s < SPLITS; ++s) {
                    sum.x += part[k][s][i].x;
                    sum.y += part[k][s][i].y;
                    sum.z += part[k][s][i].z;
                    sum.w += part[k][s][i].w;
                }
                f[4 * i] += sum.x;
                f[4 * i + 1] += sum.y;
                f[4 * i + 2] += sum.z;
                f[4 * i + 3] += sum.w;
            }
            yr[k] = V::pack(f);
        }
    }
    if (SPLITS > 0 || a.y != nullptr) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            float fx[V::N], fy[V::N], fs[V::N];
            V::unpack(xr[k], fx);
            V::unpack(yr[k], fy);
            V::unpack(sc[k], fs);
#pragma unroll
            for (int i = 0; i < V::N; ++i) fy[i] = fs[i] * fy[i];
            V::unpack(V::pack(fy), fy);
#pragma unroll
            for (int i = 0; i < V::N; ++i) fx[i] = fx[i] + fy[i];
            xr[k] = V::pack(fx);
            if (live[k] && a.sum_out != nullptr) *reinterpret_cast<uint4 *>(a.sum_out + at + (lane + 64 * k) * 16) = xr[k];
        }
    }
    if (a.norm_out == nullptr) return;
    float part = 0.f;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        float f[V::N];
        V::unpack(xr[k], f);
#pragma unroll
        for (int i = 0; i < V::N; ++i) part += f[i];          // (chunks beyond the row hold zeros)
    }
    const float mean = wave_sum(part) * a.inv_c;
    part = 0.f;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        float f[V::N];
        V::unpack(xr[k], f);
#pragma unroll
        for (int i = 0; i < V::N; ++i) {
            const float d = live[k] ? f[i] - mean : 0.f;
            part = __builtin_fmaf(d, d, part);
        }
    }
    const float rstd = 1.0f / __builtin_sqrtf(wave_sum(part) * a.inv_c + a.eps);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (!live[k]) continue;
        const int c = (lane + 64 * k) * 16;
        float f[V::N], w[V::N], b[V::N];
        V::unpack(xr[k], f);
#pragma unroll
        for (int i = 0; i < V::N; ++i) w[i] = 1.f, b[i] = 0.f;
        if (a.weight != nullptr) V::unpack(wr[k], w);
        if (a.bias != nullptr) V::unpack(br[k], b);
#pragma unroll
        for (int i = 0; i < V::N; ++i) f[i] = __builtin_fmaf((f[i] - mean) * rstd, w[i], b[i]);
        *reinterpret_cast<uint4 *>(a.norm_out + at + c) = V::pack(f);
    }
}

template <int DT, int SPLITS>
void launch(const ResidualArgs &a, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(ceil_div(a.rows, 4))), block(256);
    if (a.chunks <= 64) hipLaunchKernelGGL((residual_norm_kernel<DT, 1, SPLITS>), grid, block, 0, s, a);
    else if (a.chunks <= 128) hipLaunchKernelGGL((residual_norm_kernel<DT, 2, SPLITS>), grid, block, 0, s, a);
    else if (a.chunks <= 256) hipLaunchKernelGGL((residual_norm_kernel<DT, 4, SPLITS>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((residual_norm_kernel<DT, 8, SPLITS>), grid, block, 0, s, a);
}
template <int DT>
void launch_split(const ResidualArgs &a, int splits, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(ceil_div(a.rows, 4))), block(256);
    if (splits == 2 && a.chunks <= 64) hipLaunchKernelGGL((residual_norm_kernel<DT, 1, 2>), grid, block, 0, s, a);
    else if (splits == 2) hipLaunchKernelGGL((residual_norm_kernel<DT, 2, 2>), grid, block, 0, s, a);
    else if (a.chunks <= 64) hipLaunchKernelGGL((residual_norm_kernel<DT, 1, 4>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((residual_norm_kernel<DT, 2, 4>), grid, block, 0, s, a);
}

}  // namespace
}  // namespace come

extern "C" int come_residual_norm(const void *x, const void *y, const void *scale, int dtype, int64_t rows, int64_t channels,
                                  int64_t group_rows, int64_t group_stride, const void *weight, const void *bias, float eps,
                                  void *sum_out, void *norm_out, void *stream) {
    using namespace come;
    clear_error();
    COME_REQUIRE(dtype_ok(dtype), COME_ERR_UNSUPPORTED, "come_residual_norm: unsupported dtype %d", dtype);
    COME_REQUIRE(rows >= 0 && channels > 0, COME_ERR_INVALID, "come_residual_norm: bad sizes");
    const int64_t size = dtype_bytes(dtype), row_bytes = channels * size;
    // a wavefront holds a row: eight 16-byte chunks a lane
    COME_REQUIRE(row_bytes % 16 == 0 && row_bytes <= 8192, COME_ERR_UNSUPPORTED,
                 "come_residual_norm: rows must be a multiple of 16 bytes and at most 8 KiB (got %lld bytes)", (long long)row_bytes);
    if (rows == 0) return COME_OK;
    COME_REQUIRE(x != nullptr && (norm_out != nullptr || sum_out != nullptr), COME_ERR_INVALID, "come_residual_norm: NULL tensor");
    COME_REQUIRE(y != nullptr ? scale != nullptr : sum_out == nullptr, COME_ERR_INVALID,
                 "come_residual_norm: y, scale and sum_out go together");
    COME_REQUIRE(eps >= 0.f, COME_ERR_INVALID, "come_residual_norm: eps must be >= 0");
    COME_REQUIRE(group_rows > 0 && (group_rows >= rows || (group_stride >= group_rows * channels && group_stride * size % 16 == 0)),
                 COME_ERR_INVALID, "come_residual_norm: groups of rows overlap or are not 16-byte aligned");
    const void *aligned[] = {x, y, scale, weight, bias, sum_out, norm_out};
    for (const void *p : aligned)
        COME_REQUIRE((reinterpret_cast<uintptr_t>(p) & 15) == 0, COME_ERR_INVALID, "come_residual_norm: pointers must be 16-byte aligned");
    COME_REQUIRE(rows < (int64_t{1} << 31), COME_ERR_UNSUPPORTED, "come_residual_norm: too many rows for one launch");
    ResidualArgs a{};
    a.x = static_cast<const char *>(x);
    a.y = static_cast<const char *>(y);
    a.scale = static_cast<const char *>(scale);
    a.weight = static_cast<const char *>(weight);
    a.bias = static_cast<const char *>(bias);
    a.sum_out = static_cast<char *>(sum_out);
    a.norm_out = static_cast<char *>(norm_out);
    a.rows = rows;
    a.group_rows = group_rows;
    a.group_bytes = group_stride * size;
    a.row_bytes = row_bytes;
    a.chunks = static_cast<int>(row_bytes / 16);
    a.inv_c = 1.0f / static_cast<float>(channels);
    a.eps = eps;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == COME_F32) launch<COME_F32, 0>(a, s);
    else if (dtype == COME_BF16) launch<COME_BF16, 0>(a, s);
    else launch<COME_F16, 0>(a, s);
    COME_CHECK_LAUNCH("come_residual_norm");
    return COME_OK;
}

extern "C" int come_residual_norm_split(const void *x, const float *partial, int splits, const void *y_bias, const void *scale, int dtype,
                                        int64_t rows, int64_t channels, const void *weight, const void *bias, float eps, void *sum_out,
                                        void *norm_out, void *stream) {
    using namespace come;
    clear_error();
    COME_REQUIRE(dtype == COME_BF16 || dtype == COME_F16, COME_ERR_UNSUPPORTED, "come_residual_norm_split: only fp16 and bf16 are supported");
    COME_REQUIRE(rows >= 0 && channels > 0, COME_ERR_INVALID, "come_residual_norm_split: bad sizes");
    COME_REQUIRE(channels % 8 == 0 && channels <= 1024, COME_ERR_UNSUPPORTED,
                 "come_residual_norm_split: channels must be a multiple of 8 and at most 1024 (got %lld)", (long long)channels);
    COME_REQUIRE(splits == 2 || splits == 4, COME_ERR_INVALID, "come_residual_norm_split: 2 or 4 sums (got %d)", splits);
    if (rows == 0) return COME_OK;
    COME_REQUIRE(x != nullptr && partial != nullptr && scale != nullptr && sum_out != nullptr, COME_ERR_INVALID,
                 "come_residual_norm_split: NULL tensor");
    COME_REQUIRE(eps >= 0.f, COME_ERR_INVALID, "come_residual_norm_split: eps must be >= 0");
    const void *aligned[] = {x, partial, y_bias, scale, weight, bias, sum_out, norm_out};
    for (const void *p : aligned)
        COME_REQUIRE((reinterpret_cast<uintptr_t>(p) & 15) == 0, COME_ERR_INVALID, "come_residual_norm_split: pointers must be 16-byte aligned");
    COME_REQUIRE(rows < (int64_t{1} << 31), COME_ERR_UNSUPPORTED, "come_residual_norm_split: too many rows for one launch");
    ResidualArgs a{};
    a.x = static_cast<const char *>(x);
    a.partial = partial;
    a.y_bias = static_cast<const char *>(y_bias);
    a.scale = static_cast<const char *>(scale);
    a.weight = static_cast<const char *>(weight);
    a.bias = static_cast<const char *>(bias);
    a.sum_out = static_cast<char *>(sum_out);
    a.norm_out = static_cast<char *>(norm_out);
    a.rows = a.group_rows = rows;
    a.row_bytes = channels * 2;
    a.chunks = static_cast<int>(channels / 8);
    a.inv_c = 1.0f / static_cast<float>(channels);
    a.eps = eps;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == COME_BF16) launch_split<COME_BF16>(a, splits, s);
    else launch_split<COME_F16>(a, splits, s);
    COME_CHECK_LAUNCH("come_residual_norm_split");
    return COME_OK;
}
