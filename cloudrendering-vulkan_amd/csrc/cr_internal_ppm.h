// Internal interfaces of the photon-mapping kernels (kern_ppm.hip) used by
// cr_runtime_ppm.cpp.  Not part of the C-ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/cr/abi.h"
#include "cr_device.h"

namespace cr {

struct PpmGrid {
    const void* grid;
    int32_t nx, ny, nz, nbx, nby;
};

// A deposit as its path left it: position, power.x, direction, power.y,
// power.z, power.w.
struct PpmRecord {
    float v[12];
};
constexpr uint32_t PPM_FIRST = 8;    // record slots of every path
constexpr uint32_t PPM_CHUNK = 16;   // record slots a path takes at a time after those

struct PpmTraceArgs {
    PpmGrid g;
    cr_cloud_properties cloud;
    crd::BoxMap box;
    crd::Divisor sigmaDiv, extDiv;  // majorant in world units, maxExtinction
    cr_parameters params;
    cr_photon_map_properties pm;
    cr_render_ext ext;          // the sky the sky photons carry
    uint32_t numPaths;
    int32_t seed;
    float sunProbability;
    uint32_t maxCollisions;
    uint32_t lanes;                   // trace: lanes of each wave that take a path
    uint32_t* counts;                 // trace: deposits per path
    PpmRecord* records;               // PPM_FIRST per path, then the chunks
    uint2* chunks;                    // (path, index of its first deposit) of each chunk
    unsigned long long* chunkCount;   // trace: chunks taken (may exceed chunkCap; those past it are not stored)
    uint64_t chunkCap;
    const uint32_t* offsets;          // place: first slot of each path
    cr_photon* photons;               // place: deposits in emission order
    uint32_t* cells;                  //   their cells
    uint32_t* order;                  //   their slots (the sort's values)
};

struct PpmEstimateArgs {
    PpmGrid g;
    const float* sv;
    int32_t svx, svy, svz;
    cr_camera_properties cam;
    cr_cloud_properties cloud;
    crd::BoxMap box;
    crd::SvMap svMap;
    crd::Divisor scaleDiv, cellDiv;  // baseScaling, the photon grid's voxelSize
    cr_parameters params;
    cr_shadow_volume_properties svp;
    cr_photon_map_properties pm;
    cr_render_ext ext;
    float ambientStep;
    const uint32_t* arrivals;   // per cell
    const uint32_t* start;      // per cell: first of its run in `photons`
    const cr_photon* photons;   // deposits sorted by cell, emission order within a cell
    const float4* dirs;         // their unit directions from (theta, phi), formed when they are sorted
    const int32_t* frames;      // (seed, frameCount, pmRadius bits) per frame
    uint32_t nFrames;
    float4* image;
    int32_t W, H;
    uint32_t padded;            // 32 * (W/32 + 1), the reference's pixel-id stride
};

hipError_t launch_ppm_trace(const PpmTraceArgs& a, int dtype, int layout, hipStream_t s);
hipError_t launch_ppm_place(const PpmTraceArgs& a, uint64_t chunks, hipStream_t s);
hipError_t launch_ppm_runs(const uint32_t* keys, const uint32_t* vals, uint32_t n, uint32_t* start, uint32_t* arrivals,
                           const cr_photon* photons, cr_photon* sorted, float4* dirs, hipStream_t s);
hipError_t launch_ppm_estimate(const PpmEstimateArgs& a, int dtype, int layout, hipStream_t s);

} // namespace cr
