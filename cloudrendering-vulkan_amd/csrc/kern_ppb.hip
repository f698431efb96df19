// Photon-beam producer (shaders/PPB_PT.comp) and beam gather
// (shaders/PPB_PE.comp) for gfx950.
//
// Producer: one row of 16 lanes per sun photon path (row_walk.h).  The
// reference appends beams with atomics (PPB_PT.comp:340, :381), so its output
// order depends on timing; here the paths leave records, a scan of their
// counts gives every path its slots, and a second kernel writes beams and beam
// data there, so the arrays are a pure function of the inputs.  Corrections:
// sun photons start on the face the light enters and the face is chosen with
// if / else-if; each segment keeps its offset along the parent beam in
// _padding_beam[0].
//
// Gather: one lane per pixel; the traversal stack (64 entries, the
// reference's depth, PPB_PE.comp:414) lives in LDS but for its deepest entries; nodes are 64-B records
// holding both child boxes, so each traversal step reads one line.  The
// visit order and the order in which leaf contributions are added are the
// reference's (PPB_PE.comp:419-463).  The radiance term follows Jarosz et al.
// 2011 (beam x beam, 1D kernel) or, with refCompat, PPB_PE.comp:394-403 as
// written; boxes are tested with half their size (the reference passes the
// full size to intersectBox, PPB_PE.comp:424-431).
#include "cr_device.h"
#include "cr_internal.h"
#include "cr_internal_ppb.h"
#include "row_walk.h"

using namespace crd;

namespace {

constexpr uint32_t NONE = 0xFFFFFFFFu;
// Ceiling on delta-tracking steps of one walk along a beam (a walk through the
// unit box with majorant 64 takes ~64 steps); it only bounds the loop.
constexpr uint32_t TRACK_CEILING = 1u << 16;

template <typename T, int LAYOUT, class Map>
__device__ __forceinline__ float cloud_at(const void* grid, int32_t nx, int32_t ny, int32_t nz, int32_t nbx, int32_t nby,
                                          const Map& map, f3 p)
{
    GridView g;
    g.data = grid; g.nx = nx; g.ny = ny; g.nz = nz; g.nbx = nbx; g.nby = nby;
    return trilinear<T, LAYOUT>(g, cloud_norm(map, p));
}

// scatterRay of PPB_PT.comp:268-304 (with the final normalize).
__device__ __forceinline__ f3 scatter_norm(const cr_parameters& p, f3 n, uint32_t& rng)
{
    f3 d = scatter(p, n, rng);
    return normalize(d);
}

__device__ __forceinline__ uint32_t expand_bits10(uint32_t v)
{
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

__device__ __forceinline__ uint32_t morton30(f3 c, const float* b0, const float* b1)
{
    const float cc[3] = {c.x, c.y, c.z};
    uint32_t q[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        float n = fdiv(cc[k] - b0[k], b1[k] - b0[k]);
        q[k] = (uint32_t)fminf(fmaxf(n * 1024.0f, 0.0f), 1023.0f);
    }
    return (expand_bits10(q[0]) << 2) + (expand_bits10(q[1]) << 1) + expand_bits10(q[2]);
}

// generateSunRay's power of every photon — PPB_PT.comp:396-430 (corrected);
// `total` is the box's area seen from the sun.
__device__ __forceinline__ float photon_power(const cr::TraceArgs& a, float total)
{
    const float pdf = fdiv(1.0f, total);
    return fdiv(1.0f * a.p.lightIntensity, (float)a.p.numPaths * pdf);
}

struct SunFaces { float ax, ay, az, total; };

__device__ __forceinline__ SunFaces sun_faces(const cr::TraceArgs& a)
{
    const float* b0 = a.cloud.bounds[0];
    const float* b1 = a.cloud.bounds[1];
    const f3 L = ld3(a.p.lightDirection);
    const float dx = b1[0] - b0[0], dy = b1[1] - b0[1], dz = b1[2] - b0[2];
    SunFaces s;
    s.ax = (dz * dy) * fabsf(L.x);
    s.ay = (dx * dz) * fabsf(L.y);
    s.az = (dy * dx) * fabsf(L.z);
    s.total = (s.ax + s.ay) + s.az;
    return s;
}

// Paths firstPath .. firstPath + nPaths - 1, one per row of 16 lanes.  Every
// interaction (a stretch of beam between two collisions, or to the box's edge)
// becomes a record in an arbitrary slot of a.records; segCounts and dataCounts
// get the path's totals.  c3's trace: the paths that fill 2^22 beams took 25.6
// ms when one lane walked each path, once to count and once more to write, and
// every path of the call was counted.
template <typename T, int LAYOUT>
__global__ void __launch_bounds__(256) trace_kernel(cr::TraceArgs a)
{
    const uint32_t local = blockIdx.x * (256 / ROW) + threadIdx.x / ROW;
    if (local >= a.nPaths) return;
    const uint32_t id = a.firstPath + local;
    const RowLane R;
    uint32_t segCount = 0, dataCount = 0;
    const cr_cloud_properties& cp = a.cloud;
    if (cp.densityScaling > 0.0f) {
        const float* b0 = cp.bounds[0];
        const float* b1 = cp.bounds[1];
        uint32_t rng;
        xs_init(rng, (uint32_t)a.p.seed * id);
        const f3 L = ld3(a.p.lightDirection);
        const SunFaces F = sun_faces(a);
        const float sel = xs_float(rng) * F.total;
        const f3 c1 = mk(L.x > 0.0f ? b0[0] : b1[0], L.y > 0.0f ? b0[1] : b1[1], L.z > 0.0f ? b0[2] : b1[2]);
        f3 pos;
        {
            const float u = xs_float(rng), v = xs_float(rng);
            if (sel < F.ax) pos = mk(c1.x, b0[1] * (1.0f - u) + b1[1] * u, b0[2] * (1.0f - v) + b1[2] * v);
            else if (sel < F.ax + F.ay) pos = mk(b0[0] * (1.0f - u) + b1[0] * u, c1.y, b0[2] * (1.0f - v) + b1[2] * v);
            else pos = mk(b0[0] * (1.0f - u) + b1[0] * u, b0[1] * (1.0f - v) + b1[1] * v, c1.z);
        }
        f3 dir = L;
        const float r = a.p.radius;
        const float absorption = 1.0f - a.p.albedo;
        bool alive = a.p.maxInteractions > 0u;
        float len = 0.0f, tr = 0.0f, t = 0.0f;
        uint32_t walk = 0, rounds = 0;  // walk 0..15: transmittance distances, 16: the next collision
        if (alive) {
            float tmin = 0.0f, tmax = 0.0f;
            alive = intersect_box(b0, b1, pos, dir, tmin, tmax);
            len = length(sub(pos, add(pos, mul(dir, tmax))));
        }
        while (alive) {
            bool hit = false;
            bool end = row_walk(R, a.sigmaDiv, a.extDiv, len, t, rng, hit, [&](float d) {
                return cloud_at<T, LAYOUT>(a.grid, a.nx, a.ny, a.nz, a.nbx, a.nby, a.box, add(pos, mul(dir, d)));
            });
            if (++rounds == TRACK_CEILING / ROW) end = true;
            if (!end) continue;
            rounds = 0;
            if (walk < 16u) {
                // 16 transmittance distances — PPB_PT.comp:343-374
                if (R.i == walk) tr = t;
                t = 0.0f;
                if (++walk < 16u) continue;
                const uint32_t segs = (uint32_t)fdiv(len, r) + 1u;
                const unsigned long long slot = row_slot(R, a.recordCount);
                if (slot < a.recordCap) {
                    cr::BeamRecord& rec = a.records[slot];
                    rec.tr[R.i] = tr;
                    const float w[ROW] = {pos.x, pos.y, pos.z, len, dir.x, dir.y, dir.z, __uint_as_float(id),
                                          __uint_as_float(dataCount), __uint_as_float(segCount)};
                    float mine = w[0];
#pragma unroll
                    for (int k = 1; k < 10; k++) mine = R.i == (uint32_t)k ? w[k] : mine;
                    if (R.i < 10u) rec.head[R.i] = mine;
                }
                dataCount++;
                segCount += segs;
                continue;
            }
            // next real collision — PPB_PT.comp:473-494
            if (!hit) break;
            pos = add(pos, mul(dir, t));
            t = 0.0f;
            walk = 0;
            const float xi = xs_float(rng);
            if (!(xi > absorption)) break;
            dir = scatter_norm(a.params, dir, rng);
            if (dataCount >= a.p.maxInteractions) break;
            float tmin = 0.0f, tmax = 0.0f;
            if (!intersect_box(b0, b1, pos, dir, tmin, tmax)) break;
            len = length(sub(pos, add(pos, mul(dir, tmax))));
        }
    }
    if (R.i == 0u) {
        a.segCounts[local] = segCount;
        a.dataCounts[local] = dataCount;
    }
}

// One wave per record: its beam data and its segments, in the slots its path
// and its place on the path give it.
__device__ __forceinline__ void expand_record(const cr::TraceArgs& a, uint64_t ri, uint32_t lane)
{
    const cr::BeamRecord& rec = a.records[ri];
    const uint32_t id = __float_as_uint(rec.head[7]);
    if (id >= a.nPaths) return;
    const uint64_t segBase = a.segOffsets[id];
    if (segBase >= a.maxBeams) return;
    const uint64_t di = a.dataOffsets[id] + __float_as_uint(rec.head[8]);
    const f3 pos = mk(rec.head[0], rec.head[1], rec.head[2]), dir = mk(rec.head[4], rec.head[5], rec.head[6]);
    const float len = rec.head[3], r = a.p.radius;
    if (di < a.maxData) {
        const float power = photon_power(a, sun_faces(a).total);
        float* D = reinterpret_cast<float*>(a.data + di);
        if (lane < 20u) D[lane] = lane < 4u ? power : rec.tr[lane - 4u];
    }
    const float* b0 = a.cloud.bounds[0];
    const float* b1 = a.cloud.bounds[1];
    const uint32_t segs = (uint32_t)fdiv(len, r) + 1u;
    const float segSize = fdiv(len, (float)segs);
    const uint64_t first = segBase + __float_as_uint(rec.head[9]);
    for (uint32_t i = lane; i < segs; i += 64u) {
        const uint64_t bi = first + i;
        if (bi >= a.maxBeams) break;
        const float off = (float)i * segSize;
        const f3 st = add(pos, mul(dir, off));
        const f3 en = add(st, mul(dir, segSize));
        const uint32_t code = morton30(mk(fdiv(st.x + en.x, 2.0f), fdiv(st.y + en.y, 2.0f), fdiv(st.z + en.z, 2.0f)), b0, b1);
        uint4* B = reinterpret_cast<uint4*>(a.beams + bi);
        B[0] = make_uint4(__float_as_uint(st.x), __float_as_uint(st.y), __float_as_uint(st.z), code);
        B[1] = make_uint4(__float_as_uint(en.x), __float_as_uint(en.y), __float_as_uint(en.z), __float_as_uint(r));
        B[2] = make_uint4((uint32_t)di, __float_as_uint(off), 0u, 0u);
    }
}

// A grid dimension holds fewer than 2^32 threads and a launch beyond that runs
// only a part of them, without an error: past EXPAND_BLOCKS workgroups of four
// waves (2^22 records) the waves go on to further records.
constexpr uint32_t EXPAND_BLOCKS = 1u << 20;

__global__ void __launch_bounds__(256) expand_kernel(cr::TraceArgs a, uint64_t nRecords)
{
    for (uint64_t ri = (uint64_t)blockIdx.x * 4 + threadIdx.x / 64; ri < nRecords; ri += (uint64_t)gridDim.x * 4)
        expand_record(a, ri, threadIdx.x & 63u);
}

// A ray with a direction component exactly 0 keeps that coordinate for every
// t, so it misses every box whose slab on that axis does not hold it; the
// slab formula cannot tell (m = inf gives inf - inf = NaN, which fmaxf / fminf
// drop), so without this test such a ray culls nothing on that axis (the
// centre pixel's ray, direction (0, 0, 1), would visit the whole tree).  The
// margin covers the rounding of the center / half-size form of the box.
__device__ __forceinline__ bool outside_slab(float ro, float d, float cen, float rad)
{
    return d == 0.0f && fabsf(ro - cen) > rad + 1e-6f * (fabsf(ro) + fabsf(cen) + rad);
}

// intersectBox (PPB_PE.comp:282-300) with rad = half the box size; the box as
// center and half extent, m = 1 / rd formed once per ray; plus, for a ray
// with a zero direction component (par), the test of the axes it is parallel
// to (outside_slab is false on every axis of any other ray).
__device__ __forceinline__ bool hit_box(f3 ro, f3 rd, f3 m, bool par, const float* cen3, const float* rad3)
{
    const f3 cen = mk(cen3[0], cen3[1], cen3[2]);
    const f3 rad = mk(rad3[0], rad3[1], rad3[2]);
    const f3 n = mk(m.x * (ro.x - cen.x), m.y * (ro.y - cen.y), m.z * (ro.z - cen.z));
    const f3 k = mk(fabsf(m.x) * rad.x, fabsf(m.y) * rad.y, fabsf(m.z) * rad.z);
    const float tN = fmaxf(fmaxf(-n.x - k.x, -n.y - k.y), -n.z - k.z);
    const float tF = fminf(fminf(-n.x + k.x, -n.y + k.y), -n.z + k.z);
    bool parallelMiss = false;
    if (par)
        parallelMiss = outside_slab(ro.x, rd.x, cen.x, rad.x) || outside_slab(ro.y, rd.y, cen.y, rad.y) ||
                       outside_slab(ro.z, rd.z, cen.z, rad.z);
    return !(tN > tF || tF < 0.0f || parallelMiss);
}

// Where the camera ray passes a beam: the tests of accumulateRadiance
// (PPB_PE.comp:362-404) that decide whether the beam contributes.
struct BeamHit {
    f3 bd;       // beam direction
    f3 x;        // point of the camera ray
    float s;     // offset of the nearest point along the beam
    float dist;  // distance between them
};

__device__ __forceinline__ bool beam_hit(const cr::GatherArgs& a, const cr::SortedBeam& B, f3 ro, f3 rd, BeamHit& h)
{
    const f3 st = ld3(B.startPos), en = ld3(B.endPos);
    {
        // Skip a beam whose line passes the camera ray's line farther than its
        // radius plus a margin: the test below measures the distance between a
        // point of the camera ray and a point of the beam's line, never less
        // than the distance between the lines, so it would reject the beam too.
        // The margin (1e-4 of the coordinates' magnitude, plus 1e-3 of the
        // radius) exceeds the rounding of both computations many times over;
        // a NaN anywhere keeps the beam for the full test.
        const f3 u = sub(en, st), w = sub(st, ro);
        const f3 nrm = cross(rd, u);
        const float n2 = dot(nrm, nrm), wn = dot(w, nrm);
        const float mag = fmaxf(fmaxf(fmaxf(fabsf(ro.x), fabsf(ro.y)), fmaxf(fabsf(ro.z), fabsf(st.x))),
                                fmaxf(fmaxf(fabsf(st.y), fabsf(st.z)), fmaxf(fmaxf(fabsf(en.x), fabsf(en.y)), fabsf(en.z))));
        const float r = B.radius * 1.001f + 1e-4f * (mag + 1.0f);
        if (wn * wn > (r * r) * n2) return false;
    }
    h.bd = normalize(sub(en, st));
    if (fabsf(dot(rd, h.bd)) > 0.9f) return false;
    const f3 tangent = cross(rd, h.bd);
    const f3 pn = cross(h.bd, tangent);
    const float t = fdiv(dot(sub(st, ro), pn), dot(pn, rd));
    if (!a.refCompat && !(t >= 0.0f)) return false;
    h.x = add(ro, mul(rd, t));
    const float blen = length(sub(en, st));
    h.s = dot(sub(h.x, st), h.bd);
    if (h.s < 0.0f || h.s > blen) return false;
    const f3 proj = add(st, mul(h.bd, h.s));
    h.dist = length(sub(h.x, proj));
    return !(h.dist > B.radius);
}

// The contribution of beam bi, which beam_hit found the ray to pass.
template <typename T, int LAYOUT>
__device__ __forceinline__ void beam_radiance(const cr::GatherArgs& a, uint32_t bi, f3 ro, f3 rd, f4& acc)
{
    const cr::SortedBeam B = a.beams[bi];
    BeamHit h;
    if (!beam_hit(a, B, ro, rd, h)) return;
    const f3 bd = h.bd, x = h.x;
    const float s = h.s, dist = h.dist;
    const float q = fdiv(dist, B.radius);
    const float sq = 1.0f - q * q;
    float kern = ((15.0f / 16.0f) * sq) * sq;
    const float dens = cloud_at<T, LAYOUT>(a.grid, a.nx, a.ny, a.nz, a.nbx, a.nby, a.cloud, x);
    GridView svg;
    svg.data = a.sv; svg.nx = a.svx; svg.ny = a.svy; svg.nz = a.svz; svg.nbx = 0; svg.nby = 0;
    const float tcam = trilinear<float, LAYOUT_DENSE>(svg, sv_norm(a.svp, x));
    const cr_photon_beam_data& D = a.data[B.dataIdx];
    const float soff = a.refCompat ? s : (a.beamOff[bi] + s);
    uint32_t cnt = 0;
#pragma unroll
    for (int i = 0; i < 16; i++)
        if (D.trDistances[i] >= soff) cnt++;
    const float tb = fdiv((float)cnt, 16.0f);
    const f3 nrd = neg(rd);
    const float ph = phase_pdf(a.params, bd, nrd);
    const float cosA = dot(bd, nrd);
    float sinA, sc;
    if (a.refCompat) {
        sinA = 1.0f - cosA * cosA;
        sc = dens;
    } else {
        kern = fdiv(kern, B.radius);
        sinA = fsqrt(1.0f - cosA * cosA);
        sc = a.albedo * fdiv(dens * a.cloud.densityScaling, a.cloud.baseScaling);
    }
    const float w = fdiv(ph, sinA);
    const float ks = kern * sc;
    acc.x = acc.x + (((ks * D.power[0]) * tcam) * tb) * w;
    acc.y = acc.y + (((ks * D.power[1]) * tcam) * tb) * w;
    acc.z = acc.z + (((ks * D.power[2]) * tcam) * tb) * w;
    acc.w = acc.w + (((ks * D.power[3]) * tcam) * tb) * w;
}

constexpr int GATHER_THREADS = 128;
constexpr uint32_t STACK = 64;      // traversal stack entries (the reference's depth), the first
constexpr uint32_t STACK_LDS = 24;  //   of them in LDS, deeper ones in scratch memory
// Beams a lane found while walking the tree wait in two short queues, so that
// the wave runs the beam tests and the radiance for many lanes at once (one
// leaf in seven visited nodes is tested and a quarter of those contribute:
// run where they were found, most of the wave waited for a few lanes).  Both
// queues are first in, first out, so a ray's contributions are added in the
// order of the reference's traversal.  1080p frame over 2^22 beams: 26.1 ms
// with the tests in the walk, 12.6 with the queues, and 8.5 with 16 instead of
// 32 lanes to start a stage, four waves per SIMD and 8x8 instead of 16x4
// pixels per wave (stages at 8, 24, 32 or 48 lanes, queues of 16, and 3 or 5
// waves are within 3% or slower); under other suns such frames take 9.2-11.1.
constexpr uint32_t FOUND = 8, PASSED = 4;                    // queue lengths (powers of two)
constexpr uint32_t FOUND_LANES = 16, PASSED_LANES = 16;      // lanes with work that start a stage
template <typename T, int LAYOUT>
__global__ void __launch_bounds__(GATHER_THREADS, 4) gather_kernel(cr::GatherArgs a)
{
    // entry e of a lane's array at [e * GATHER_THREADS]: bank-conflict free
    __shared__ uint32_t stack_mem[STACK_LDS * GATHER_THREADS];
    __shared__ uint32_t found_mem[FOUND * GATHER_THREADS];
    __shared__ uint32_t passed_mem[PASSED * GATHER_THREADS];
    uint32_t* stack = stack_mem + threadIdx.x;
    uint32_t* found = found_mem + threadIdx.x;
    uint32_t* passed = passed_mem + threadIdx.x;
    uint32_t deep[STACK - STACK_LDS];
    // a wave takes 8x8 pixels
    const int32_t x = (int32_t)(blockIdx.x * 16 + (threadIdx.x >> 6) * 8 + (threadIdx.x & 7));
    const int32_t y = (int32_t)(blockIdx.y * 8 + ((threadIdx.x >> 3) & 7));
    const bool inside = x < a.W && y < a.H;
    uint32_t visited = 0, tested = 0, rays = 0;
    if (inside) {
        float4 o = a.image[(size_t)y * a.W + x];
        f4 acc;
        acc.x = o.x; acc.y = o.y; acc.z = o.z; acc.w = o.w;
        const uint32_t id = (uint32_t)x + (uint32_t)y * a.padded;
        for (uint32_t f = 0; f < a.nFrames; f++) {
            const int32_t seed = a.frames[2 * f];
            const uint32_t fc = (uint32_t)a.frames[2 * f + 1];
            float dx = (float)(x - a.cam.halfWidth), dy = (float)(y - a.cam.halfHeight);
            if (a.jitter) {
                uint32_t rng;
                xs_init(rng, (uint32_t)seed * id);
                dx = dx + (xs_float(rng) - 0.5f);
                dy = dy + (xs_float(rng) - 0.5f);
            }
            f3 ro, rd;
            camera_ray(a.cam, dx, dy, ro, rd);
            rays++;
            f4 L;
            L.x = 0.0f; L.y = 0.0f; L.z = 0.0f; L.w = 0.0f;
            const f3 m = mk(fdiv(1.0f, rd.x), fdiv(1.0f, rd.y), fdiv(1.0f, rd.z));
            const bool par = rd.x == 0.0f || rd.y == 0.0f || rd.z == 0.0f;
            if (a.n == 1) {
                // (lo + hi) / 2: halving is exact, so * 0.5 is the same value
                const float cen[3] = {(a.leafLo[0] + a.leafHi[0]) * 0.5f, (a.leafLo[1] + a.leafHi[1]) * 0.5f,
                                      (a.leafLo[2] + a.leafHi[2]) * 0.5f};
                const float rad[3] = {(a.leafHi[0] - a.leafLo[0]) * 0.5f, (a.leafHi[1] - a.leafLo[1]) * 0.5f,
                                      (a.leafHi[2] - a.leafLo[2]) * 0.5f};
                if (hit_box(ro, rd, m, par, cen, rad)) {
                    beam_radiance<T, LAYOUT>(a, 0, ro, rd, L);
                    tested++;
                }
            } else if (a.n > 1) {
                const uint32_t inner = a.n - 1;
                uint32_t sp = 0;  // entries on the stack
                uint32_t cur = 0;
                uint32_t f0 = 0, nf = 0, p0 = 0, np = 0;  // the queues' first entries and lengths
                // every internal node is visited at most once per ray; the
                // bound only protects against a malformed tree
                uint32_t budget = a.n;
                for (;;) {
                    const uint32_t nPassed = (uint32_t)__popcll(__ballot(np > 0u));
                    const bool canTest = nf > 0u && np < PASSED;
                    const uint32_t nTest = (uint32_t)__popcll(__ballot(canTest));
                    const bool canWalk = cur != NONE && nf + 2u <= FOUND;
                    const uint32_t nWalk = (uint32_t)__popcll(__ballot(canWalk));
                    if (nPassed >= PASSED_LANES || (nPassed && !nTest && !nWalk)) {
                        if (np > 0u) {
                            const uint32_t bi = passed[p0 * GATHER_THREADS];
                            p0 = (p0 + 1u) & (PASSED - 1u);
                            np--;
                            beam_radiance<T, LAYOUT>(a, bi, ro, rd, L);
                        }
                    } else if (nTest >= FOUND_LANES || (nTest && !nWalk)) {
                        if (canTest) {
                            const uint32_t bi = found[f0 * GATHER_THREADS];
                            f0 = (f0 + 1u) & (FOUND - 1u);
                            nf--;
                            BeamHit h;
                            if (beam_hit(a, a.beams[bi], ro, rd, h)) {
                                passed[((p0 + np) & (PASSED - 1u)) * GATHER_THREADS] = bi;
                                np++;
                            }
                        }
                    } else if (nWalk) {
                        if (canWalk) {
                            if (budget-- == 0u || cur >= inner) {
                                atomicOr(a.overflow, 2u);
                                cur = NONE;
                                sp = 0;
                            } else {
                                visited++;
                                const cr::TravNode nd = a.nodes[cur];
                                const bool hl = hit_box(ro, rd, m, par, nd.cen[0], nd.rad[0]);
                                const bool hr = hit_box(ro, rd, m, par, nd.cen[1], nd.rad[1]);
                                const bool ll = (nd.leafMask & 1u) != 0, lr = (nd.leafMask & 2u) != 0;
                                // the node's hit leaves, left before right
                                if (hl && ll) {
                                    found[((f0 + nf) & (FOUND - 1u)) * GATHER_THREADS] = nd.child[0] - inner;
                                    nf++;
                                    tested++;
                                }
                                if (hr && lr) {
                                    found[((f0 + nf) & (FOUND - 1u)) * GATHER_THREADS] = nd.child[1] - inner;
                                    nf++;
                                    tested++;
                                }
                                const bool tl = hl && !ll, tr = hr && !lr;
                                if (!tl && !tr) {
                                    if (sp == 0u) {
                                        cur = NONE;
                                    } else {
                                        sp--;
                                        cur = sp < STACK_LDS ? stack[sp * GATHER_THREADS] : deep[sp - STACK_LDS];
                                    }
                                } else {
                                    cur = tl ? nd.child[0] : nd.child[1];
                                    if (tl && tr) {
                                        // the reference's stack holds a sentinel in its first entry
                                        if (sp < STACK - 1u) {
                                            if (sp < STACK_LDS) stack[sp * GATHER_THREADS] = nd.child[1];
                                            else deep[sp - STACK_LDS] = nd.child[1];
                                            sp++;
                                        } else {
                                            atomicOr(a.overflow, 1u);
                                        }
                                    }
                                }
                            }
                        }
                    } else {
                        break;
                    }
                }
            }
            // running mean — PPB_PE.comp:482-486
            const float nn = (float)fc;
            const float d = (float)(fc + 1u);
            acc.x = fdiv(L.x + acc.x * nn, d);
            acc.y = fdiv(L.y + acc.y * nn, d);
            acc.z = fdiv(L.z + acc.z * nn, d);
            acc.w = fdiv(L.w + acc.w * nn, d);
        }
        float4 o2;
        o2.x = acc.x; o2.y = acc.y; o2.z = acc.z; o2.w = acc.w;
        a.image[(size_t)y * a.W + x] = o2;
    }
    const unsigned long long s0 = wave_sum_u64(rays), s1 = wave_sum_u64(visited), s2 = wave_sum_u64(tested);
    if ((threadIdx.x & 63) == 0) {
        unsigned long long* const cnt =
            a.counters + ((blockIdx.x + blockIdx.y * gridDim.x) % cr::COUNTER_SLOTS) * cr::COUNTER_STRIDE;
        atomicAdd(cnt + 0, s0);
        atomicAdd(cnt + 1, s1);
        atomicAdd(cnt + 2, s2);
    }
}

} // namespace

namespace cr {

hipError_t launch_trace(const TraceArgs& a, int dtype, int layout, hipStream_t s)
{
    if (a.nPaths == 0) return hipSuccess;
    const dim3 g((a.nPaths + 256 / ROW - 1) / (256 / ROW));
    if (dtype == CR_DTYPE_F16) {
        if (layout == LAYOUT_BRICK4) hipLaunchKernelGGL((trace_kernel<__half, LAYOUT_BRICK4>), g, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((trace_kernel<__half, LAYOUT_DENSE>), g, dim3(256), 0, s, a);
    } else {
        if (layout == LAYOUT_BRICK4) hipLaunchKernelGGL((trace_kernel<float, LAYOUT_BRICK4>), g, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((trace_kernel<float, LAYOUT_DENSE>), g, dim3(256), 0, s, a);
    }
    return hipGetLastError();
}

hipError_t launch_trace_expand(const TraceArgs& a, uint64_t records, hipStream_t s)
{
    if (records == 0) return hipSuccess;
    const uint64_t blocks = (records + 3) / 4;
    hipLaunchKernelGGL(expand_kernel, dim3((unsigned)(blocks < EXPAND_BLOCKS ? blocks : EXPAND_BLOCKS)), dim3(256), 0, s, a, records);
    return hipGetLastError();
}

hipError_t launch_gather(const GatherArgs& a, int dtype, int layout, hipStream_t s)
{
    dim3 g((unsigned)((a.W + 15) / 16), (unsigned)((a.H + 7) / 8));
    if (dtype == CR_DTYPE_F16) {
        if (layout == LAYOUT_BRICK4) hipLaunchKernelGGL((gather_kernel<__half, LAYOUT_BRICK4>), g, dim3(GATHER_THREADS), 0, s, a);
        else hipLaunchKernelGGL((gather_kernel<__half, LAYOUT_DENSE>), g, dim3(GATHER_THREADS), 0, s, a);
    } else {
        if (layout == LAYOUT_BRICK4) hipLaunchKernelGGL((gather_kernel<float, LAYOUT_BRICK4>), g, dim3(GATHER_THREADS), 0, s, a);
        else hipLaunchKernelGGL((gather_kernel<float, LAYOUT_DENSE>), g, dim3(GATHER_THREADS), 0, s, a);
    }
    return hipGetLastError();
}

} // namespace cr
