// adjoint.h — launch parameters of the path-replay adjoint kernels.
#pragma once
#include "context.h"

// The differentiable Path estimator: path.rgen:26-104 without roulette,
// direct lighting on, spp samples per pixel (sample k uses the RNG frame
// word k ^ seed), over `variants` texel sets that replace the scene textures
// aid (albedo, rgb) and rid (roughness).
//
// Work items: item i covers variant i % variants of pixel p = i / variants,
// pixels ordered by 8x8 tiles (tile p / 64, row-major inside), so one wave
// holds the variants of few pixels.  Those lanes trace the same rays until a
// glossy sample on a variant surface separates them, and their gradient
// scatters go to different variants' arrays.
struct AdjLaunch {
    float inv_view[16];
    float inv_projection[16];
    uint32_t width, height;
    int32_t max_depth;
    uint32_t spp, seed, variants;
    float sky_col[3];
    int32_t aid, rid;          // replaced scene textures (-1: none)
    uint32_t aw, ah, rw, rh;   // their texel grids
    uint32_t tiles_x;
    uint32_t n_items;          // tiles * 64 * variants
    uint32_t rec_depth;        // bounces per sample in the cache's path records (0: none)
    uint32_t run;              // groups of 64 items a wave takes at once (launch_adjoint sets it)
    uint32_t texel_step;       // floats between a texel's channels: 1, or the variants if interleaved (launch_adjoint)
    uint32_t trunk_depth;      // forward: bounces of a sample whose rays the variants share (0: none)
};

// The forward shares a sample's rays between its variants from this many
// variants on (8 variants of 400x300, 16 samples: 10.8 -> 9.5 ms forward and
// backward; 4 of 512x512, 8 samples: 13.5 ms with and without), and up to
// this many bounces.
constexpr uint32_t kAdjTrunkMinVariants = 8;
constexpr uint32_t kAdjTrunkMaxDepth = 16;
constexpr uint32_t kAdjTrunkMinGroups = 4;  // groups of 64 items per wave
constexpr uint64_t kAdjTrunkMinLanes = 48;  // lanes of the shared walk in use
inline uint32_t adj_trunk_depth(int32_t max_depth, uint32_t variants) {
    if (variants < kAdjTrunkMinVariants) return 0u;
    return max_depth < (int32_t)kAdjTrunkMaxDepth ? (uint32_t)max_depth : kAdjTrunkMaxDepth;
}
// records of the shared rays per wave (16 B each)
inline size_t adj_trunk_words4(uint32_t trunk_depth) { return (size_t)trunk_depth * 4u * 64u; }

// Bounces per sample the sample cache records (3 flag bits per bounce in one
// 32-bit word), and the cache's size in floats: per sample the radiance (3),
// and with records two 16-byte hit records per bounce (the path's closest
// hit and the NEE MIS ray's) and the flag word.
constexpr uint32_t kAdjRecMaxDepth = 10;
inline uint32_t adj_rec_depth(int32_t max_depth) {
    return max_depth >= 1 && max_depth <= (int32_t)kAdjRecMaxDepth ? (uint32_t)max_depth : 0u;
}
inline size_t adj_cache_floats(uint32_t spp, uint32_t n_items, uint32_t rec_depth) {
    return (size_t)spp * n_items * (3u + (rec_depth ? 8u * rec_depth + 1u : 0u));
}

// Device arrays of one call (all row-major, float32):
//   albedo [V][ah][aw][3], rough [V][rh][rw]       variant texels
//   images [V][H][W][3]                            forward output
//   cache  [spp][3][n_items]                        per-sample radiance (optional)
//   d_images [V][H][W][3]                          adjoint of images
//   g_albedo, g_rough like albedo, rough           texel gradients (overwritten)
struct AdjBuffers {
    const float* albedo;
    const float* rough;
    float* images;
    float* cache;
    const float* d_images;
    float* g_albedo;
    float* g_rough;
};

// Floats of the interleaved texels and their gradients (0: the kernels use the
// caller's arrays).  The variants of a pixel sit in neighbouring lanes and
// read the same texels, each of its own texture: 64 cache lines per load and,
// in the backward, per atomic.  With the variants interleaved (texel, channel,
// variant) neighbouring lanes read and add to neighbouring words: 512x512, 32
// variants of 256x256 texels, 8 samples: backward 25.5 -> 21.5 ms, forward
// 31.4 -> 30.8.  It costs a transpose of the texels per call (and of the
// gradients), about 30 us each there, so only where the samples outnumber the
// texels.
constexpr uint32_t kAdjInterleaveMinVariants = 4;
constexpr size_t kAdjInterleaveMaxBytes = (size_t)4 << 30;
inline size_t adj_texel_floats(uint64_t pixels, uint32_t spp, uint32_t variants, uint64_t texels_a, uint64_t texels_r) {
    const uint64_t n = 2u * variants * (3u * texels_a + texels_r);
    if (variants < kAdjInterleaveMinVariants || texels_a + texels_r > pixels * spp) return 0;
    return n * sizeof(float) <= kAdjInterleaveMaxBytes ? (size_t)n : 0;
}

// What an adjoint keeps on the device between calls.
struct AdjWork {
    uint32_t* work;   // persistent-grid work counter
    uint32_t* spill;  // traversal stack spill of the resident threads
    uint4* trunk;     // shared rays of the forward, per wave; nullptr: no sharing
    float* texels;    // interleaved texels and gradients; nullptr: the caller's arrays
    uint32_t blocks;  // most workgroups of a launch; spill and trunk are sized for them
};

// workgroups of the adjoint kernels: what the chip holds at once (or the
// tuning's count, if lower)
uint32_t adjoint_blocks(lt_context* ctx);
// counts: NULL, or kCountSlots u64 that the counting kernel variants fill
lt_status launch_adjoint(lt_context* ctx, const AdjLaunch& L, const AdjBuffers& B, bool backward, const AdjWork& W,
                         unsigned long long* counts, hipStream_t stream);
