// How the path tracer's passes are cut into work items and launches: host
// arithmetic only, without HIP.
#pragma once

#include <stdint.h>

namespace cr {

constexpr uint32_t PT_FEW_FRAMES = 16;

// Frames per work item of a chunked pass: at least `perLane` items per resident
// lane while there are samples to make them of, each of at most `most` samples.
// Renders: chunks of 4 measured best where samples abound (a 16-job batch: 125 ms
// with chunks of up to 16, 101 with 8, 85 with 4, 95 with 1; 512x512 at 128 spp:
// 26.0, -, 20.6, 23.4), and 8 items per lane where they do not (256x256 at 64
// spp: 3.18 ms; with 4 items 3.47, with 32 3.32).
// Record passes, whose samples are short, pay for the set-up of more items: whole
// learned renders with 2, 4 and 8 items per lane take 7.47, 7.50 and 7.90 ms at
// 1080p and 8 spp, 4.97, 5.02 and 5.87 at 4 spp, 6.43, 6.18 and 6.06 at 1280x720
// and 16 spp, 3.43, 3.06 and 3.56 at 640x360 and 32 spp (chunks of 16 everywhere
// 7.47, 5.00, 6.47 and 3.83, and 1.76 ms at 128x128 and 32 spp against 0.57);
// chunks of more than 16 are not needed, 32 spp at 1080p 27.7 ms with 16, 29.0
// with 4.
constexpr uint32_t PT_CHUNK_RENDER = 4, PT_ITEMS_RENDER = 8;
constexpr uint32_t PT_CHUNK_RECORD = 16, PT_ITEMS_RECORD = 4;
static_assert(PT_CHUNK_RENDER <= PT_FEW_FRAMES && PT_CHUNK_RECORD <= PT_FEW_FRAMES, "chunked items are few-frame items");
inline uint32_t pt_chunk(uint64_t pixels, uint32_t samples, uint64_t lanes, uint32_t perLane, uint32_t most)
{
    const uint64_t c = pixels * samples / (perLane * lanes);
    return (uint32_t)(c < 1 ? 1 : (c > most ? most : c));
}

// Workgroups of 256 lanes for `items` work items, at most `resident`, the
// number the chip holds at a time, and at least one.
inline int pt_blocks(uint64_t items, int resident)
{
    const uint64_t needed = items / 256u + (items % 256u != 0u);
    if (needed < (uint64_t)(resident > 0 ? resident : 1)) return needed ? (int)needed : 1;
    return resident > 0 ? resident : 1;
}

// Samples stored by one chunked launch at most (4 GiB); more go in several
// launches, each of which ends on its longest paths (16-job batch: 88.6 ms
// with 1 GiB).
constexpr uint64_t PT_SAMPLE_BUDGET = 1ull << 28;

// Frames (or continuations) that a launch has to hold for storing its samples to
// be worth it: with room for 1, 2, 4, 16 and 64 of them a render takes 17.1, 9.0,
// 5.4, 2.9 and 2.4 ms at 256x256 and 64 spp and 160, 122, 131, 94 and 82 at 1080p
// (brick tracking), one cloud's training data 275, 133, 68, 27 and 12.5; whole
// pixels (or records), which need no room, 11.4, 127 and 156.
constexpr uint32_t PT_LEAST_STORED = 2;

// The number of samples there is room for, by alloc(n), which takes memory for n
// of them or returns false: as near to `want` as halving (and what was held
// before, `had`) comes, at least `least`, or 0.
template <class Alloc>
uint64_t pt_sample_room(uint64_t want, uint64_t least, uint64_t had, Alloc alloc)
{
    for (uint64_t n = want; !alloc(n);) {
        if (n <= least) return 0;
        uint64_t next = n / 2;
        if (had < n && next < had) next = had;
        n = next > least ? next : least;
        want = n;
    }
    return want;
}

} // namespace cr
