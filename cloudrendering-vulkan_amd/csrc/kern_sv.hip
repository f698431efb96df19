// Shadow-volume precompute (shaders/ShadowVolume.comp, dispatched by
// RenderTechniqueSV::RecordDrawCommands, RenderTechniqueSV.cpp:102-113).
//
// Along each light-space column (x, y) T(x,y,z) = exp(-voxelSize * sum_{k<=z}
// sigma(p_k)), accumulated exactly as ShadowVolume.comp:84-93 states it
// (exp(-accumulatedDistance * accumulatedValue / (z + 1))).  Consecutive
// lanes own consecutive x, so every z-slice access is a coalesced row.
// With per-axis texel counts (extension) the lattice spacing along axis k is
// voxelSize * (N - 1) / (N_k - 1), N = voxelAxisCount; the cubic default is
// the reference lattice.
#include "cr_device.h"
#include "cr_internal.h"

using namespace crd;

namespace {

// The lattice point's density in world units; false outside the cloud.
template <typename T, int LAYOUT>
__device__ __forceinline__ bool lattice_sigma(const cr::SVArgs& a, int32_t x, int32_t y, int32_t z, float& v)
{
    GridView g;
    g.data = a.grid; g.nx = a.nx; g.ny = a.ny; g.nz = a.nz; g.nbx = a.nbx; g.nby = a.nby;
    const cr_shadow_volume_properties& P = a.svp;
    const float fx = (float)x * a.k[0], fy = (float)y * a.k[1], fz = (float)z * a.k[2];
    f3 p;
    p.x = P.bounds[0][0] + ((fx * P.right[0] + fy * P.up[0]) + fz * P.lightDirection[0]) * P.voxelSize;
    p.y = P.bounds[0][1] + ((fx * P.right[1] + fy * P.up[1]) + fz * P.lightDirection[1]) * P.voxelSize;
    p.z = P.bounds[0][2] + ((fx * P.right[2] + fy * P.up[2]) + fz * P.lightDirection[2]) * P.voxelSize;
    if (!in_box(a.cloud.bounds[0], a.cloud.bounds[1], p)) return false;
    v = div1(a.scaleDiv, trilinear<T, LAYOUT, true>(g, cloud_norm(a.box, p)) * a.cloud.densityScaling);
    return true;
}

// Many columns: one lane each, in one pass.
template <typename T, int LAYOUT>
__global__ void __launch_bounds__(256) sv_kernel(cr::SVArgs a)
{
    const int32_t x = (int32_t)(blockIdx.x * 64 + (threadIdx.x & 63));
    const int32_t y = (int32_t)(blockIdx.y * 4 + (threadIdx.x >> 6));
    if (x >= a.dx || y >= a.dy) return;
    const float hz = a.svp.voxelSize * a.k[2];
    float acc = 0.0f, accDist = 0.0f;
    const size_t plane = (size_t)a.dx * (size_t)a.dy;
    float* out = a.out + (size_t)x + (size_t)a.dx * (size_t)y;
    for (int32_t z = 0; z < a.dz; z++) {
        float v;
        if (lattice_sigma<T, LAYOUT>(a, x, y, z, v)) acc = acc + v;
        accDist = accDist + hz;
        out[(size_t)z * plane] = crd_expf(fdiv((-accDist) * acc, (float)((uint32_t)z + 1u)));
    }
}

// Few columns: sigma at the lattice points first, every point by itself (0 outside
// the cloud, which leaves a column's sum as it is), then the columns' sums.
template <typename T, int LAYOUT>
__global__ void __launch_bounds__(256) sv_sample_kernel(cr::SVArgs a)
{
    const int32_t x = (int32_t)(blockIdx.x * 64 + (threadIdx.x & 63));
    const int32_t y = (int32_t)(blockIdx.y * 4 + (threadIdx.x >> 6));
    if (x >= a.dx || y >= a.dy) return;
    const size_t plane = (size_t)a.dx * (size_t)a.dy;
    float* out = a.out + (size_t)x + (size_t)a.dx * (size_t)y;
    for (int32_t z = (int32_t)blockIdx.z; z < a.dz; z += (int32_t)gridDim.z) {
        float v;
        if (!lattice_sigma<T, LAYOUT>(a, x, y, z, v)) v = 0.0f;
        out[(size_t)z * plane] = v;
    }
}

// The columns' running sums, AHEAD texels fetched together.
__global__ void __launch_bounds__(64) sv_sum_kernel(cr::SVArgs a)
{
    constexpr int AHEAD = 16;
    const uint32_t c = blockIdx.x * 64u + threadIdx.x, plane = (uint32_t)a.dx * (uint32_t)a.dy;
    if (c >= plane) return;
    const float hz = a.svp.voxelSize * a.k[2];
    float acc = 0.0f, accDist = 0.0f;
    float* out = a.out + c;
    for (int32_t z0 = 0; z0 < a.dz; z0 += AHEAD) {
        float v[AHEAD];
#pragma unroll
        for (int k = 0; k < AHEAD; k++) v[k] = z0 + k < a.dz ? out[(size_t)(z0 + k) * plane] : 0.0f;
#pragma unroll
        for (int k = 0; k < AHEAD; k++) {
            acc = acc + v[k];
            accDist = accDist + hz;
            if (z0 + k < a.dz)
                out[(size_t)(z0 + k) * plane] = crd_expf(fdiv((-accDist) * acc, (float)((uint32_t)(z0 + k) + 1u)));
        }
    }
}

} // namespace

namespace cr {

constexpr uint32_t SPLIT_COLUMNS = 163840;  // 2.5 waves per SIMD

hipError_t launch_sv(const SVArgs& a, int dtype, int layout, hipStream_t s)
{
    // One lane per column leaves the chip idle while columns are few, and each lane
    // waits for its lookups one after the other; two passes cost the texels' extra
    // trip to memory.  Cubes on an FP32 128^3 grid, one pass and two: 64 58 and 32
    // us, 256 220 and 139, 384 327 and 262, 448 389 and 392, 512 469 and 664; on a
    // 320^3 grid 256 292 and 195, 500 993 and 1229.
    const uint32_t plane = (uint32_t)a.dx * (uint32_t)a.dy;
    const bool split = plane < SPLIT_COLUMNS;
    dim3 grid((unsigned)((a.dx + 63) / 64), (unsigned)((a.dy + 3) / 4));
    if (split) grid.z = (unsigned)(a.dz < 65535 ? a.dz : 65535);
#define CR_SV(T, L)                                                                                 \
    do {                                                                                            \
        if (split) hipLaunchKernelGGL((sv_sample_kernel<T, L>), grid, dim3(256), 0, s, a);          \
        else hipLaunchKernelGGL((sv_kernel<T, L>), grid, dim3(256), 0, s, a);                       \
    } while (0)
    if (dtype == CR_DTYPE_F16) {
        if (layout == LAYOUT_BRICK4) CR_SV(__half, LAYOUT_BRICK4);
        else CR_SV(__half, LAYOUT_DENSE);
    } else {
        if (layout == LAYOUT_BRICK4) CR_SV(float, LAYOUT_BRICK4);
        else CR_SV(float, LAYOUT_DENSE);
    }
#undef CR_SV
    if (split) hipLaunchKernelGGL(sv_sum_kernel, dim3((plane + 63u) / 64u), dim3(64), 0, s, a);
    return hipGetLastError();
}

} // namespace cr
