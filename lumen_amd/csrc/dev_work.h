// dev_work.h — how the waves of a persistent grid share a range of items.
//
// Atomics on one address are served one after another, about 11 ns each
// whichever XCD they come from (2.07M rays taken 16 at a time from one counter:
// 130k atomics, 1.44 ms; 64 at a time: 0.35 ms of a 0.64 ms query pass).  A
// counter that every wave adds to for every few items is therefore what
// bounds a kernel of a few milliseconds.  So the items are cut into tiles of
// 64; most tiles are dealt out beforehand, round robin over the waves, and only
// the rest, which evens out the waves' uneven costs, come from the counter, a
// whole tile per atomic.  A range of at most one tile per wave needs no
// counter at all.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dev_math.h"

namespace ltd {

// Per cent of the tiles dealt out beforehand (at least one round).  Ray
// batches, BDPT, VCM and SPPM lose 1-4 % with 45 (2.07M bounce rays 624 ->
// 633 us, SPPM 13.9 -> 14.5 ms) and more with 25.  Images of paths and of
// texture variants (`image` below) have dear and cheap regions that a wave's
// dealt tiles may keep hitting: 60 -> 45 takes 16 Path frames of 509x383 from
// 1.79 to 1.62 ms and the adjoint at 512x512 from 53.0 to 49.0 ms (90 %: 72
// ms), and a 1080p Path frame is even.
constexpr uint32_t kStaticPct = 60;
constexpr uint32_t kStaticPctImage = 45;

// Rounds of one tile per wave that need no counter.
__host__ __device__ inline uint32_t static_rounds(uint32_t n_tiles, uint32_t n_waves, bool image) {
    const uint32_t r = (uint32_t)((uint64_t)n_tiles * (image ? kStaticPctImage : kStaticPct) / 100u / n_waves);
    return r ? r : 1u;
}

// Workgroups of `waves_per_block` waves for n_items: at most `blocks`, and no
// more than the tiles need, in multiples of 8 (the XCDs) where that leaves
// at least one round.
inline uint32_t work_blocks(uint64_t n_items, uint32_t blocks, uint32_t waves_per_block) {
    const uint64_t tiles = (n_items + 63u) / 64u, need = (tiles + waves_per_block - 1u) / waves_per_block;
    const uint64_t up = (need + 7u) / 8u * 8u;
    return (uint32_t)(up < blocks ? up : blocks);
}
// true if that grid takes tiles from the counter, which must then start at zero
inline bool work_counted(uint64_t n_items, uint32_t blocks, uint32_t waves_per_block, bool image = false) {
    const uint32_t tiles = (uint32_t)((n_items + 63u) / 64u), waves = blocks * waves_per_block;
    return static_rounds(tiles, waves, image) * (uint64_t)waves < tiles;
}

// The wave's part of the items; every field is wave-uniform.
struct WaveTiles {
    uint32_t next;      // its next dealt tile
    uint32_t stride;    // waves of the grid
    uint32_t n_static;  // tiles dealt out beforehand
    uint32_t n_tiles, n_items;
    uint32_t base, left;  // items of its current tile not handed out yet
    bool done;            // no tile is left
    uint32_t* work;       // counter of the tiles beyond n_static, zero at the launch
};

// Call with the whole wave active.  Workgroups are dealt to the 8 XCDs round
// robin (blockIdx mod 8), each with its own L2: the waves of one XCD are
// numbered consecutively, so that a round gives it one run of tiles.  Where
// regions of an image differ in cost that would give one XCD, or one CU, all
// the dear ones: with `image` neighbouring tiles go to different workgroups
// instead (a 160x120 preview frame 252 -> 237 us; the adjoint at 256x200, 3
// variants: 5.12 -> 3.93 ms; a 1080p Path frame even).
LT_DEV WaveTiles wave_tiles(uint32_t n_items, uint32_t* work, bool image = false) {
    WaveTiles t;
    const uint32_t wpb = blockDim.x >> 6, wib = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    t.stride = gridDim.x * wpb;
    if (image)
        t.next = wib * gridDim.x + blockIdx.x;
    else
        t.next = (gridDim.x & 7u) == 0u ? ((blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3)) * wpb + wib
                                    : blockIdx.x * wpb + wib;
    t.n_items = n_items;
    t.n_tiles = (n_items + 63u) >> 6;
    t.n_static = static_rounds(t.n_tiles, t.stride, image) * t.stride;
    t.base = t.left = 0u;
    t.done = false;
    t.work = work;
    return t;
}

// Moves on to the wave's next tile; false (and done) if there is none.  The
// whole wave must be active.
LT_DEV bool next_tile(WaveTiles& t) {
    uint32_t tile;
    if (t.next < t.n_static) {
        tile = t.next;
        t.next += t.stride;
    } else {
        uint32_t k = 0u;
        if ((threadIdx.x & 63u) == 0u && t.n_static < t.n_tiles) k = atomicAdd(t.work, 1u);
        tile = t.n_static + (uint32_t)__builtin_amdgcn_readfirstlane((int)k);
    }
    t.done = tile >= t.n_tiles;
    t.base = tile << 6;
    t.left = t.done ? 0u : min(64u, t.n_items - t.base);
    return !t.done;
}

// Hands the lanes of `idle` (wave-uniform mask) an item each, in lane order,
// from the current tile and, where that runs out, the next one: true and the
// lane's item, or false (not idle, or nothing left for it now).  The whole
// wave must be active.
LT_DEV bool take_items(WaveTiles& t, unsigned long long idle, uint32_t& item) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t rank = (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
    const bool want = ((idle >> lane) & 1ull) != 0ull;
    uint32_t need = (uint32_t)__popcll(idle), given = 0u;
    bool got = false;
    while (need != 0u) {
        if (t.left == 0u && (t.done || !next_tile(t))) break;
        const uint32_t n = min(need, t.left);
        if (want && rank >= given && rank < given + n) {
            item = t.base + (rank - given);
            got = true;
        }
        t.base += n;
        t.left -= n;
        given += n;
        need -= n;
    }
    return got;
}

}  // namespace ltd
