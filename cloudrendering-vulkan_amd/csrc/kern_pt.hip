// Launches of the path tracer: the single-job render and the batched render.
#include "pt_kernel.h"

#include <algorithm>

namespace {

// PathTracer.comp:420-424
__device__ __forceinline__ void blend_sample(float4& acc, float4 L, uint32_t fc)
{
    const float n = (float)fc, d = (float)(fc + 1u);
    acc.x = fdiv(L.x + acc.x * n, d);
    acc.y = fdiv(L.y + acc.y * n, d);
    acc.z = fdiv(L.z + acc.z * n, d);
    acc.w = fdiv(L.w + acc.w * n, d);
}

// The running mean of the stored samples of pixel p, in frame order, blended
// into the image.
__device__ __forceinline__ void blend_pixel(const cr::PTArgs& a, uint32_t pixels, uint32_t p)
{
    float4 acc = a.image[p];
#pragma unroll 4
    for (uint32_t f = 0; f < a.nFrames; f++)
        blend_sample(acc, a.samples[(size_t)f * pixels + p], (uint32_t)a.frames[2 * f + 1]);
    a.image[p] = acc;
}

// One workgroup per square of 8x8 tiles.  A pixel that misses the box shows the
// background in every frame and is finished here; masks[square] gets the tiles
// with a pixel that hits it.
__global__ void __launch_bounds__(256) squares_kernel(cr::PTArgs a, uint32_t sqX, unsigned long long* masks)
{
    __shared__ uint32_t sky;
    __shared__ unsigned long long mask;
    if (threadIdx.x == 0) { sky = 0u; mask = 0ull; }
    __syncthreads();
    const uint32_t lane = lane_id(), sq = blockIdx.x, tilesY = ((uint32_t)a.H + 7u) >> 3;
    uint32_t skyPixels = 0;
    for (uint32_t k = threadIdx.x >> 6; k < 64u; k += 4u) {
        const uint32_t tx = (sq % sqX) * 8u + (k & 7u), ty = (sq / sqX) * 8u + (k >> 3);
        if (tx >= a.tilesX || ty >= tilesY) continue;
        const int32_t x = (int32_t)(tx * 8u + (lane & 7u)), y = (int32_t)(ty * 8u + (lane >> 3));
        const bool inside = x < a.W && y < a.H;
        f3 pos, dir;
        const bool miss = inside && camera_entry(a, x, y, pos, dir);
        const bool hit = __ballot(inside && !miss) != 0ull;
        if (lane == 0 && hit) atomicOr(&mask, 1ull << k);
        if (miss) {
            skyPixels++;
            const f4 bg = background(a.ext, dir);
            const float4 L = make_float4(bg.x, bg.y, bg.z, bg.w);
            float4* px = a.image + (size_t)y * a.W + x;
            float4 acc = *px;
            for (uint32_t f = 0; f < a.nFrames; f++) blend_sample(acc, L, (uint32_t)a.frames[2 * f + 1]);
            *px = acc;
        }
    }
    if (skyPixels) atomicAdd(&sky, skyPixels);
    __syncthreads();
    if (threadIdx.x == 0) {
        masks[sq] = mask;
        if (sky) {
            const unsigned long long paths = (unsigned long long)sky * a.nFrames;
            unsigned long long* const cnt = a.counters + (sq % cr::COUNTER_SLOTS) * cr::COUNTER_STRIDE;
            atomicAdd(cnt + 0, paths);
            atomicAdd(cnt + 1, paths);
        }
    }
}

// The list from the squares' masks: square r goes to part r mod 8; one wave per
// part, one lane per square.
__global__ void __launch_bounds__(512) list_kernel(const unsigned long long* masks, uint32_t squares, uint32_t sqX,
                                                   uint32_t tilesX, uint32_t* list, uint32_t* starts)
{
    __shared__ uint32_t total[8];
    const uint32_t lane = lane_id(), part = threadIdx.x >> 6;
    const uint32_t mine = squares > part ? (squares - part + 7u) / 8u : 0u;  // squares of this part
    uint32_t n = 0;
    for (uint32_t j = lane; j < mine; j += 64u) n += (uint32_t)__popcll(masks[part + 8u * j]);
    for (int off = 32; off >= 1; off >>= 1) n += (uint32_t)__shfl_xor((int)n, off, 64);
    if (lane == 0) total[part] = n;
    __syncthreads();
    uint32_t at = 0;
    for (uint32_t k = 0; k < part; k++) at += total[k];
    if (lane == 0) starts[part] = at;
    if (threadIdx.x == 511u) starts[8] = at + total[7];
    for (uint32_t j0 = 0; j0 < mine; j0 += 64u) {
        const uint32_t j = j0 + lane, sq = j < mine ? part + 8u * j : 0u;
        unsigned long long m = j < mine ? masks[sq] : 0ull;
        const uint32_t c = (uint32_t)__popcll(m);
        uint32_t incl = c;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)incl, off, 64);
            if (lane >= (uint32_t)off) incl += o;
        }
        uint32_t w = at + incl - c;
        while (m) {
            const uint32_t k = (uint32_t)__ffsll((long long)m) - 1u;
            m &= m - 1ull;
            list[w++] = ((sq / sqX) * 8u + (k >> 3)) * tilesX + (sq % sqX) * 8u + (k & 7u);
        }
        at += (uint32_t)__shfl((int)incl, 63, 64);
    }
}

__global__ void __launch_bounds__(256) blend_kernel(cr::PTArgs a)
{
    const uint32_t p = blockIdx.x * 256 + threadIdx.x, pixels = (uint32_t)a.W * (uint32_t)a.H;
    if (p >= pixels) return;
    f3 pos, dir;
    if (camera_entry(a, (int32_t)(p % (uint32_t)a.W), (int32_t)(p / (uint32_t)a.W), pos, dir)) return;  // see squares_kernel
    blend_pixel(a, pixels, p);
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
    if (p < pixels && J.samples) blend_pixel(J, pixels, p);
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

// Layout of `lists`: the squares' masks (2 words each), the list, the nine part starts.
static uint64_t list_squares(const PTArgs& a) { return (uint64_t)((a.W + 63) / 64) * (uint64_t)((a.H + 63) / 64); }
uint64_t pt_list_starts(const PTArgs& a) { return 2u * list_squares(a) + a.totalIdx / 64u; }
uint64_t pt_list_words(const PTArgs& a) { return pt_list_starts(a) + 9u; }

hipError_t launch_pt_list(const PTArgs& a, uint32_t* lists, hipStream_t s)
{
    const uint32_t n = (uint32_t)list_squares(a), sqX = (uint32_t)(a.W + 63) / 64u;
    unsigned long long* masks = reinterpret_cast<unsigned long long*>(lists);
    hipLaunchKernelGGL(squares_kernel, dim3(n), dim3(256), 0, s, a, sqX, masks);
    hipLaunchKernelGGL(list_kernel, dim3(1), dim3(512), 0, s, masks, n, sqX, a.tilesX, lists + 2u * n,
                       lists + pt_list_starts(a));
    return hipGetLastError();
}

hipError_t launch_pt_blend(const PTArgs& a, hipStream_t s)
{
    const uint32_t pixels = (uint32_t)a.W * (uint32_t)a.H;
    hipLaunchKernelGGL(blend_kernel, dim3((pixels + 255) / 256), dim3(256), 0, s, a);
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

hipError_t launch_pt(const PTArgs& a, int dtype, int layout, int blocks, int cus, hipStream_t s)
{
    // No more than a wave per SIMD: workgroups of one wave, dealt over the whole
    // chip, where four neighbouring tiles of one workgroup would share a CU (256x256
    // at 64 spp, brick tracking 58.4 -> 55.5 ms, 128x128 at 32 spp with the shadow
    // volume 5.8 -> 5.4; beyond that neighbours sharing a cache are worth more,
    // 512x512 at 64 spp 16.9 ms against 21.7), and the kernel of whole pixels however
    // few their frames (256x256 with the shadow volume, 4 frames 0.94 -> 0.80 ms, one
    // frame 0.27 -> 0.24).
    const bool sparse = blocks <= cus && !a.samples;
    if (a.chunk <= PT_FEW_FRAMES && !sparse) return launch_pt_few(a, dtype, layout, blocks, s);
    BatchArgs none = {};
    if (sparse) blocks = (int)std::min<uint32_t>(4u * (uint32_t)blocks, (a.totalIdx + 63u) / 64u);
    return launch(pick<false, K_RENDER>(dtype, layout, a.ext.trackingMode, a.ext.neeMode), a, none, blocks, sparse ? 64 : 256, 0, s);
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
