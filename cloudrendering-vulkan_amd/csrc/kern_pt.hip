// Launches of the path tracer: the single-job render and the batched render.
#include "pt_kernel.h"

#include "cr_internal_ppb.h"

namespace {

__global__ void __launch_bounds__(256) order_keys_kernel(const uint32_t* cost, uint32_t n, uint32_t* keys, uint32_t* vals)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    keys[i] = ~cost[i];
    vals[i] = i;
}

// The running mean of nf stored samples of pixel p, in frame order
// (PathTracer.comp:420-424), blended into the image.
__device__ __forceinline__ void blend_pixel(const float4* samples, const int32_t* frames, uint32_t nf, float4* image,
                                            uint32_t pixels, uint32_t p)
{
    float4 acc = image[p];
#pragma unroll 4
    for (uint32_t f = 0; f < nf; f++) {
        const float4 L = samples[(size_t)f * pixels + p];
        const uint32_t fc = (uint32_t)frames[2 * f + 1];
        const float n = (float)fc, d = (float)(fc + 1u);
        acc.x = fdiv(L.x + acc.x * n, d);
        acc.y = fdiv(L.y + acc.y * n, d);
        acc.z = fdiv(L.z + acc.z * n, d);
        acc.w = fdiv(L.w + acc.w * n, d);
    }
    image[p] = acc;
}

__global__ void __launch_bounds__(256) blend_kernel(const float4* samples, const int32_t* frames, uint32_t nf, float4* image,
                                                    uint32_t pixels)
{
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    if (p < pixels) blend_pixel(samples, frames, nf, image, pixels, p);
}

// The jobs of one batched launch; a job's workgroups start at its blendBase
// (a job that blends in the path tracer has none).
__global__ void __launch_bounds__(256) blend_batch_kernel(cr::BatchArgs b)
{
    uint32_t lo = 0, hi = b.nJobs - 1u;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1u) >> 1;
        if (b.jobs[mid].blendBase <= blockIdx.x) lo = mid;
        else hi = mid - 1u;
    }
    const cr::PTArgs& J = b.jobs[lo];
    const uint32_t pixels = (uint32_t)J.W * (uint32_t)J.H;
    const uint32_t p = (blockIdx.x - J.blendBase) * 256 + threadIdx.x;
    if (p < pixels && J.samples) blend_pixel(J.samples, J.frames, J.nFrames, J.image, pixels, p);
}

// out[r] = ((0 + sample 0) + sample 1) + ..., over `total` samples at the end;
// ns samples per launch, accumulated in `out` between launches.
__global__ void __launch_bounds__(64) sum_kernel(const float4* samples, const float* points, uint32_t m, uint32_t ns,
                                                 uint32_t sample0, uint32_t total, float4* out)
{
    const uint32_t r = blockIdx.x * 64 + threadIdx.x;
    if (r >= m) return;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (points[(size_t)r * 8 + 7] > 0.5f) {
        if (sample0) acc = out[r];
#pragma unroll 8
        for (uint32_t s = 0; s < ns; s++) {
            const float4 v = samples[(size_t)s * m + r];
            acc.x = acc.x + v.x;
            acc.y = acc.y + v.y;
            acc.z = acc.z + v.z;
            acc.w = acc.w + v.w;
        }
        if (sample0 + ns == total) {
            const float n = (float)total;
            acc = make_float4(fdiv(acc.x, n), fdiv(acc.y, n), fdiv(acc.z, n), fdiv(acc.w, n));
        }
    }
    out[r] = acc;
}

} // namespace

namespace cr {

hipError_t launch_pt_blend(const PTArgs& a, hipStream_t s)
{
    const uint32_t pixels = (uint32_t)a.W * (uint32_t)a.H;
    hipLaunchKernelGGL(blend_kernel, dim3((pixels + 255) / 256), dim3(256), 0, s, a.samples, a.frames, a.nFrames, a.image,
                       pixels);
    return hipGetLastError();
}

hipError_t launch_pt_blend_batch(const BatchArgs& b, uint32_t blocks, hipStream_t s)
{
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL(blend_batch_kernel, dim3(blocks), dim3(256), 0, s, b);
    return hipGetLastError();
}

hipError_t launch_pt_sum(const PTArgs& a, uint32_t total, hipStream_t s)
{
    hipLaunchKernelGGL(sum_kernel, dim3((a.nPoints + 63) / 64), dim3(64), 0, s, a.samples, a.points, a.nPoints, a.spp,
                       a.sample0, total, a.out);
    return hipGetLastError();
}

uint32_t pt_order_counts(uint32_t n) { return sort_counts_words(n) * 4u; }

hipError_t launch_tile_order(const uint32_t* cost, uint32_t n, uint32_t* keys, uint32_t* vals, uint32_t* keys_tmp,
                             uint32_t* vals_tmp, uint32_t* counts, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(order_keys_kernel, dim3((n + 255) / 256), dim3(256), 0, s, cost, n, keys, vals);
    return launch_radix_sort(keys, vals, keys_tmp, vals_tmp, counts, n, s);
}

hipError_t launch_pt(const PTArgs& a, int dtype, int layout, int blocks, hipStream_t s)
{
    if (a.chunk <= PT_FEW_FRAMES) return launch_pt_few(a, dtype, layout, blocks, s);
    BatchArgs none = {};
    return launch(pick<false, K_RENDER>(dtype, layout, a.ext.trackingMode, a.ext.neeMode), a, none, blocks, 256, 0, s);
}

int pt_blocks_per_cu(int dtype, int layout, uint32_t tracking, uint32_t nee, uint32_t chunk)
{
    if (chunk <= PT_FEW_FRAMES) return pt_few_blocks_per_cu(dtype, layout, tracking, nee);
    return occupancy(pick<false, K_RENDER>(dtype, layout, tracking, nee), 256, 0);
}

hipError_t launch_pt_batch(const BatchArgs& b, int dtype, int layout, uint32_t tracking, uint32_t nee, int blocks,
                           int block_threads, hipStream_t s)
{
    PTArgs none = {};
    return launch(pick<true, K_RENDER>(dtype, layout, tracking, nee), none, b, blocks, block_threads,
                  (size_t)b.nJobs * sizeof(PTArgs), s);
}

int pt_batch_blocks_per_cu(int dtype, int layout, uint32_t tracking, uint32_t nee, int block_threads, uint32_t n_jobs)
{
    return occupancy(pick<true, K_RENDER>(dtype, layout, tracking, nee), block_threads, (size_t)n_jobs * sizeof(PTArgs));
}

} // namespace cr
