// Per-Gaussian features to packed rows and back.
//
// The packed layout (one row per visible (b, c, g), gsplat/cuda/csrc/
// ProjectionEWA3DGSPacked.cu:234-284) makes rasterization() gather
// per-Gaussian features into rows -- opacities[batch_ids, gaussian_ids],
// colors[batch_ids, gaussian_ids] (gsplat/rendering.py:782, 170-213) -- and
// autograd scatter the row gradients back with index_put(accumulate=True),
// which PyTorch runs as a sort plus a segmented sum.
//
// Both directions here are driven by Gaussian through the inverse map
// row_of[(b C + c) N + g] (packed row or -1) that the packed projection
// writes: the gather reads each Gaussian's feature row once and stores it to
// its rows; the scatter sums a Gaussian's row gradients over the C cameras in
// camera order and writes its gradient row once (zeros when it is visible
// nowhere).  Deterministic, no atomics, no zero fill; consecutive threads
// take consecutive Gaussians, so the per-Gaussian streams are coalesced.
#include "common.h"

namespace gs {
namespace {

constexpr int kRowsThreads = 256;

__global__ void __launch_bounds__(kRowsThreads)
    rows_gather_kernel(int64_t B, int64_t C, int64_t N, int F,
                       const float *__restrict__ src,
                       const int32_t *__restrict__ row_of,
                       float *__restrict__ out) {
    const int64_t bg = (int64_t)blockIdx.x * kRowsThreads + threadIdx.x;
    if (bg >= B * N)
        return;
    const int64_t b = bg / N, g = bg - b * N;
    const float *s = src + bg * F;
    for (int64_t c = 0; c < C; ++c) {
        const int32_t r = row_of[(b * C + c) * N + g];
        if (r < 0)
            continue;
        float *o = out + (int64_t)r * F;
        for (int f = 0; f < F; ++f)
            o[f] = s[f];
    }
}

template <int F>
__global__ void __launch_bounds__(kRowsThreads)
    rows_scatter_kernel_fixed(int64_t B, int64_t C, int64_t N,
                              const int32_t *__restrict__ row_of,
                              const float *__restrict__ v_out,
                              float *__restrict__ v_src) {
    const int64_t bg = (int64_t)blockIdx.x * kRowsThreads + threadIdx.x;
    if (bg >= B * N)
        return;
    const int64_t b = bg / N, g = bg - b * N;
    float acc[F];
#pragma unroll
    for (int f = 0; f < F; ++f)
        acc[f] = 0.f;
    for (int64_t c = 0; c < C; ++c) {
        const int32_t r = row_of[(b * C + c) * N + g];
        if (r < 0)
            continue;
#pragma unroll
        for (int f = 0; f < F; ++f)
            acc[f] += v_out[(int64_t)r * F + f];
    }
#pragma unroll
    for (int f = 0; f < F; ++f)
        v_src[bg * F + f] = acc[f];
}

// From four features on, one thread per (Gaussian, feature): a wave reads and
// writes whole lines, where one thread per Gaussian strode over its row (32
// features, 111,785 Gaussians, 14 MB each way: scatter 49.3 -> 14.1 us, gather
// 23.3 -> 11.4 us).  The cameras are summed in the same order.
template <bool SCATTER>
__global__ void __launch_bounds__(kRowsThreads)
    rows_wide_kernel(int64_t B, int64_t C, int64_t N, int F,
                     const int32_t *__restrict__ row_of,
                     const float *__restrict__ in, float *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * kRowsThreads + threadIdx.x;
    if (i >= B * N * F)
        return;
    // 32-bit division where the index allows it
    const int64_t bg = i <= 0xffffffffll ? (int64_t)((uint32_t)i / (uint32_t)F) : i / F;
    const int f = (int)(i - bg * F);
    const int64_t b = B == 1 ? 0 : bg / N, g = bg - b * N;
    float v = SCATTER ? 0.f : in[i];
    for (int64_t c = 0; c < C; ++c) {
        const int32_t r = row_of[(b * C + c) * N + g];
        if (r < 0)
            continue;
        if (SCATTER)
            v += in[(int64_t)r * F + f];
        else
            out[(int64_t)r * F + f] = v;
    }
    if (SCATTER)
        out[i] = v;
}

// one thread per value: four features or more, as far as a grid reaches
bool rows_wide(int64_t n, int32_t F) {
    return F >= 4 && ceil_div(n * F, kRowsThreads) < (1ll << 31);
}

int rows_check(int64_t B, int64_t C, int64_t N, int32_t F, const int32_t *row_of) {
    GS_REQUIRE(B >= 0 && C >= 0 && N >= 0 && F >= 0, "rows: negative size");
    if (B * C * N > 0)
        GS_REQUIRE(row_of != nullptr, "rows: NULL row_of");
    return GSPLAT_OK;
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" int gsplat_rows_gather(int64_t B, int64_t C, int64_t N, int32_t F,
                                  const float *src, const int32_t *row_of,
                                  float *out, gsplat_stream_t stream) {
    clear_error();
    GS_TRY(rows_check(B, C, N, F, row_of));
    if (B * N == 0 || C == 0 || F == 0)
        return GSPLAT_OK;
    GS_REQUIRE(src && out, "rows_gather: NULL buffer");
    const bool wide = rows_wide(B * N, F);
    const unsigned grid = (unsigned)ceil_div(wide ? B * N * F : B * N, kRowsThreads);
    if (wide)
        rows_wide_kernel<false><<<grid, kRowsThreads, 0, as_stream(stream)>>>(
            B, C, N, F, row_of, src, out);
    else
        rows_gather_kernel<<<grid, kRowsThreads, 0, as_stream(stream)>>>(B, C, N, F, src,
                                                                        row_of, out);
    return check_launch("rows_gather_kernel");
}

extern "C" int gsplat_rows_scatter_sum(int64_t B, int64_t C, int64_t N,
                                       int32_t F, const int32_t *row_of,
                                       const float *v_out, float *v_src,
                                       gsplat_stream_t stream) {
    clear_error();
    GS_TRY(rows_check(B, C, N, F, row_of));
    if (B * N == 0 || F == 0)
        return GSPLAT_OK;
    GS_REQUIRE(v_src != nullptr && (C == 0 || v_out != nullptr),
               "rows_scatter_sum: NULL buffer");
    const unsigned grid = (unsigned)ceil_div(B * N, kRowsThreads);
    hipStream_t st = as_stream(stream);
    switch (F) {
    case 1:
        rows_scatter_kernel_fixed<1><<<grid, kRowsThreads, 0, st>>>(B, C, N, row_of, v_out, v_src);
        break;
    case 3:
        rows_scatter_kernel_fixed<3><<<grid, kRowsThreads, 0, st>>>(B, C, N, row_of, v_out, v_src);
        break;
    case 2:
        rows_scatter_kernel_fixed<2><<<grid, kRowsThreads, 0, st>>>(B, C, N, row_of, v_out, v_src);
        break;
    default:
        GS_REQUIRE(rows_wide(B * N, F), "rows_scatter_sum: more than 2^39 values");
        rows_wide_kernel<true><<<(unsigned)ceil_div(B * N * F, kRowsThreads), kRowsThreads, 0,
                                 st>>>(B, C, N, F, row_of, v_out, v_src);
        break;
    }
    return check_launch("rows_scatter_kernel");
}
