// Delta-tracking walks by rows of 16 lanes, for the photon-beam producer.
//
// A photon path is one chain of random numbers: where a walk ends decides from
// which draw the next one goes on, so paths are serial and a trace of some
// thousand paths is bound by the latency of one step (logarithm, division,
// eight-tap lookup), not by throughput.  But until a walk ends, its draws do
// not depend on what it meets: step i takes draw 2i for its free flight and
// draw 2i + 1 for its collision test.  So the 16 lanes of a row take the next
// 16 steps of one path's walk together: each jumps the xorshift state ahead to
// its draws (the generator is linear over GF(2): 32 columns of its (2i)-th
// power per lane), the flight distances are added in step order by a lane
// shift, all lookups go out at once, and the first lane whose step leaves the
// segment or collides ends the walk; the steps past it are dropped and the
// state is the one after the last draw the walk used.  Same draws, same sums
// in the same order as one lane stepping alone.  A path of the producer makes
// 17 walks of some twenty steps per interaction; photon mapping's paths, whose
// walks end after two or three steps in dense cloud, gain nothing from this
// (12 800 paths 1.03 ms, one lane each 0.97; a million 50 ms against 4.9).
#pragma once

#include "cr_device.h"

namespace crd {

constexpr int ROW = 16;

struct RowJumps { uint32_t m[ROW][32]; };

// m[i][b]: the state xorshift32 reaches from 1 << b after 2 i draws.
constexpr RowJumps make_row_jumps()
{
    RowJumps j{};
    for (int b = 0; b < 32; b++) {
        uint32_t s = 1u << b;
        for (int i = 0; i < ROW; i++) {
            j.m[i][b] = s;
            for (int k = 0; k < 2; k++) {
                s ^= s << 13;
                s ^= s >> 17;
                s ^= s << 5;
            }
        }
    }
    return j;
}
static __device__ const RowJumps row_jumps = make_row_jumps();

struct RowLane {
    uint32_t i;        // lane of the row
    uint32_t jump[32];

    __device__ __forceinline__ RowLane() : i(threadIdx.x & (ROW - 1))
    {
#pragma unroll
        for (int b = 0; b < 32; b++) jump[b] = row_jumps.m[i][b];
    }
    // The state 2 i draws after s.
    __device__ __forceinline__ uint32_t ahead(uint32_t s) const
    {
        uint32_t r = 0;
#pragma unroll
        for (int b = 0; b < 32; b++) r ^= (uint32_t)((int32_t)(s << (31 - b)) >> 31) & jump[b];
        return r;
    }
};

// A slot of a shared list for the row, counted by its first lane.
__device__ __forceinline__ unsigned long long row_slot(const RowLane& R, unsigned long long* count)
{
    unsigned long long slot = 0;
    if (R.i == 0u) slot = atomicAdd(count, 1ull);
    return __shfl(slot, 0, ROW);
}

// One round of a walk: up to 16 steps from distance t and state rng (both the
// same in all lanes of the row).  Returns true when the walk ended, with t the
// distance of its last step, hit whether it collided there (else it left the
// segment) and rng the state after its last draw; otherwise t and rng are
// those after 16 steps.  `density`: the cloud's density at a distance.
template <class Density>
__device__ __forceinline__ bool row_walk(const RowLane& R, const Divisor& sigmaBar, const Divisor& maxExtinction, float len, float& t,
                                         uint32_t& rng, bool& hit, Density density)
{
    uint32_t s = R.ahead(rng);
    const float zeta = xs_float(s);
    const uint32_t afterFlight = s;
    const float xi = xs_float(s);
    const float d = div1(sigmaBar, -crd_logf(zeta));
    // t + d of the row's first lane, then lane by lane (row_shr:1)
    float at = t;
#pragma unroll
    for (int k = 0; k < ROW; k++)
        at = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(t), __float_as_int(at), 0x111, 0xf, 0xf, false)) + d;
    const bool left = !(at <= len);
    bool stop = left;
    if (!left) stop = xi < div1(maxExtinction, density(at));
    const uint32_t row = (threadIdx.x & 63u) & ~(uint32_t)(ROW - 1);
    const uint32_t ends = (uint32_t)(__ballot(stop) >> row) & 0xffffu;
    const int last = ends ? (int)__ffs((int)ends) - 1 : ROW - 1;
    t = __shfl(at, last, ROW);
    const uint32_t after = left ? afterFlight : s;
    rng = (uint32_t)__shfl((int)after, last, ROW);
    hit = !(t <= len) ? false : ends != 0u;
    return ends != 0u;
}

} // namespace crd
