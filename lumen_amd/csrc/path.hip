// path.hip — the Path integrator on gfx950 (persistent form).
//
// Persistent lanes with path regeneration over the samples of a launch's
// frames, dealt out in 8x8 pixel tiles (k_path_regen).  The samples of several
// frames go to a buffer that k_path_mean folds in frame order into the
// reference's running mean (path.rgen:106-112), so the result equals
// frame-by-frame launches; a single frame's go straight into the mean.
// Per-sample logic: src/shaders/integrators/path/path.rgen:26-104 and
// src/shaders/integrators/pt_commons.glsl:3-47.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "context.h"
#include "dev_scene.h"
#include "dev_atmosphere.h"
#include "dev_nee.h"
#include "dev_trace.h"
#include "path.h"

using namespace ltd;

namespace {

// The state of one path between bounces (path.rgen:26-100).  The hit
// payload is not part of it: a bounce's closest-hit trace either fills every
// field or misses and ends the path, so only the NEE MIS ray of the same
// bounce sees a stale payload (ray.rmiss:13), which nee_sample records.
struct PathState {
    RNG seed;
    f3 origin, direction, throughput, col;
    uint32_t pix;
    int depth;
    bool last_specular;
};

LT_DEV void path_start(const PathLaunch& L, uint32_t x, uint32_t y, uint32_t frame_word, PathState& p) {
    p.seed = {x, y, frame_word, 0u};
    const float r0 = rnd(p.seed);
    const float r1 = rnd(p.seed);
    const float jx = r0 - 0.5f, jy = r1 - 0.5f;
    const float ux = ((float)x + 0.5f + jx) / (float)L.width, uy = ((float)y + 0.5f + jy) / (float)L.height;
    const float dx = ux * 2.0f - 1.0f, dy = uy * 2.0f - 1.0f;
    const f4 o4 = mul4(L.inv_view, f4{0.0f, 0.0f, 0.0f, 1.0f});
    const f4 tg = mul4(L.inv_projection, f4{dx, dy, 1.0f, 1.0f});
    const f3 tn = normalize(mk3(tg.x, tg.y, tg.z));
    const f4 d4 = mul4(L.inv_view, f4{tn.x, tn.y, tn.z, 0.0f});
    p.origin = {o4.x, o4.y, o4.z};
    p.direction = {d4.x, d4.y, d4.z};
    p.col = mk3(0.0f);
    p.throughput = mk3(1.0f);
    p.last_specular = false;
    p.depth = 0;
}

// one iteration of path.rgen:46-100; returns false when the path has ended.
// The bounce draws its random numbers in the reference's order (NEE light
// sample, NEE BSDF sample, continuation, Russian roulette), then traces its
// NEE rays, whose terms use the throughput before the continuation.
template <bool COUNT>
LT_DEV bool path_bounce(const SceneView& sv, const PathLaunch& L, PathState& p, const TraceStack& stk, Ctr& c) {
    NeeRays nee;
    bool alive = true, has_nee = false;
    {
        Payload hp;
        trace_closest<COUNT>(sv, p.origin, p.direction, stk, hp, c);
        if (!hp.valid) {
            if (p.depth > 0 || L.direct_lighting == 1)
                p.col += p.throughput * sky_radiance(sv, ld3(L.sky_col), p.origin, p.direction, PATH_TMAX);
            return false;
        }
        const Mat hit_mat = load_material(sv, hp.material_idx, hp.uv);
        if ((p.depth == 0 && L.direct_lighting == 1) || p.last_specular) p.col += p.throughput * hit_mat.emissive;
        if (p.depth >= L.max_depth - 1) return false;
        const f3 wo = -p.direction;
        f3 n_s = hp.n_s;
        bool side = true;
        f3 n_g = hp.n_g;
        if (dot(hp.n_g, wo) < 0.0f) n_g = -n_g;
        if (dot(n_g, hp.n_s) < 0.0f) {
            n_s = -n_s;
            side = false;
        }
        p.origin = offset_ray(hp.pos, n_g);
        p.last_specular = is_specular(hit_mat);
        if (!p.last_specular && (p.depth > 0 || L.direct_lighting == 1)) {
            nee_sample(sv, p.seed, hit_mat, hp, side, n_s, wo, p.throughput, L.nee_pick, nee);
            has_nee = true;
        }
        float pdf, cos_theta;
        const float s0 = rnd(p.seed), s1 = rnd(p.seed), s2 = rnd(p.seed);
        const f3 f = sample_bsdf(n_s, wo, hit_mat, 1, side, p.direction, pdf, cos_theta, s0, s1, s2);
        if (pdf == 0.0f) {
            alive = false;
        } else {
            const f3 thr = p.throughput * (f * fabsf(cos_theta) / pdf);
            float rr_scale = 1.0f;
            if (hit_mat.bsdf_props & LT_BSDF_FLAG_TRANSMISSION) rr_scale *= side ? 1.0f / hit_mat.ior : hit_mat.ior;
            if (p.depth > RR_MIN_DEPTH) {
                const float rr_prob = fminf(0.95f, luminance(thr) * rr_scale);
                if (rr_prob == 0.0f || rr_prob < rnd(p.seed)) alive = false;
                else p.throughput = thr / rr_prob;
            } else {
                p.throughput = thr;
            }
        }
    }
    if (has_nee) p.col += nee_trace<COUNT>(sv, nee, stk, c);
    p.depth++;
    return alive;
}

// Four waves per SIMD (128 VGPRs; the path state across a traversal spills to
// scratch, which stays in cache): 6.5 ms per 1080p terrain frame against
// 9.0 ms at the unconstrained 203 VGPRs / 2 waves, in an earlier form.
#ifndef LT_PATH_MEGA_WAVES
#define LT_PATH_MEGA_WAVES 4
#endif

// Path regeneration (the persistent form): each lane runs one bounce of its
// path per iteration and, once the path ends, takes the next sample, so paths
// of uneven length (Russian roulette, escapes) never leave lanes idle until
// the longest path of a tile ends.  Per path the arithmetic, the RNG stream
// and the result are those of path_sample.
//
// The items are the samples of L.spp frames, tile by tile of 8x8 pixels and a
// tile's frames one after another: the frames share one launch, so the chip
// drains once and not once per frame, and an image of fewer pixels than the
// chip has lanes still fills it.  With one frame a sample goes straight into
// the running mean; with more it goes to `rad` and k_path_mean folds a pixel's
// samples in frame order.  16 frames of the 1080p terrain with a launch and a
// contended counter each: 57.0 ms, in one launch 48.1 ms; of a 509 x 383 Cornell
// box 4.2 (a wave per tile and its 16 samples in lockstep) and 1.8 ms.
template <bool COUNT>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(LT_PATH_MEGA_WAVES))) void k_path_regen(
    SceneView sv, PathLaunch L, float4* __restrict__ accum, float4* __restrict__ rad, uint32_t* __restrict__ work,
    uint32_t* __restrict__ spill, unsigned long long* __restrict__ counts) {
    __shared__ uint32_t s_stack[ltb::kLdsWords * kTraceBlock];
    const uint32_t gtid = blockIdx.x * blockDim.x + threadIdx.x;
    TraceStack stk{s_stack + threadIdx.x, spill + (size_t)gtid * (ltb::kStackTotal - ltb::kLdsStack)};
    const uint32_t tiles_x = (L.width + 7) / 8, tiles_y = (L.height + 7) / 8;
    const uint32_t n_items = tiles_x * tiles_y * L.spp * 64u;
    const uint32_t frame0 = L.frame_dev ? *L.frame_dev : L.frame_start;
    Ctr c{0, 0, 0, 0};
    PathState p;
    bool has = false;
    WaveTiles wt = wave_tiles(n_items, work, true);
    for (;;) {
        const unsigned long long idle = __ballot(!has);
        const uint32_t n_idle = (uint32_t)__popcll(idle);
        if (n_idle == 64u || (!wt.done && n_idle >= L.regen_min)) {
            if (n_idle == 64u && wt.done) break;
            uint32_t t = 0u;
            if (take_items(wt, idle, t)) {
                const uint32_t w = t & 63u;
                uint32_t tile = t >> 6, f = 0u;
                if (L.spp > 1u) {
                    f = tile % L.spp;
                    tile /= L.spp;
                }
                const uint32_t x = (tile % tiles_x) * 8 + (w & 7u), y = (tile / tiles_x) * 8 + (w >> 3);
                if (x < L.width && y < L.height) {
                    path_start(L, x, y, (frame0 + f) ^ L.seed, p);
                    p.pix = f * (L.width * L.height) + y * L.width + x;
                    has = true;
                }
            }
        }
        if (has && !path_bounce<COUNT>(sv, L, p, stk, c)) {
            has = false;
            const bool ok = !isnan(luminance(p.col));  // path.rgen:102-104
            if (L.spp > 1u) {
                rad[p.pix] = make_float4(p.col.x, p.col.y, p.col.z, ok ? 1.0f : 0.0f);
            } else if (ok) {
                float4 acc = accum[p.pix];
                accumulate_mean(acc, p.col.x, p.col.y, p.col.z, frame0);
                accum[p.pix] = acc;
            }
        }
    }
    if (COUNT) flush_counts(c, counts);
}

// folds the samples of a multi-frame launch into the running mean (HBM bound:
// 16 B per sample)
__global__ __launch_bounds__(256) void k_path_mean(const float4* __restrict__ rad, float4* __restrict__ accum,
                                                   uint32_t n, uint32_t frame0, uint32_t frames) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 acc = accum[i];
    for (uint32_t f = 0; f < frames; f++) {
        const float4 r = rad[(size_t)f * n + i];
        if (r.w != 0.0f) accumulate_mean(acc, r.x, r.y, r.z, frame0 + f);
    }
    accum[i] = acc;
}

__global__ void k_zero_u32(uint32_t* p, uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

}  // namespace

// workgroups of a persistent kernel: the tuning's count, but no more than the
// chip holds at once (the tiles dealt out beforehand must all be under way)
static size_t path_blocks(lt_context* ctx, const void* kernel) {
    return (size_t)ctx->num_cus * std::min(ctx->tuning.path_blocks_per_cu, resident_blocks(kernel, 0u));
}

void path_samples_free(PathSamples& s) {
    if (s.rad) (void)hipFree(s.rad);
    s = PathSamples{};
}

lt_status launch_path_persistent(lt_context* ctx, PathSamples& ps, const PathLaunch& L0, float4* accum, int count,
                                 uint64_t* d_counts) {
    const size_t blocks = path_blocks(ctx, count ? reinterpret_cast<const void*>(&k_path_regen<true>)
                                                 : reinterpret_cast<const void*>(&k_path_regen<false>));
    lt_status st = ensure_spill(ctx, blocks * kTraceBlock);
    if (st != LT_OK) return st;
    if (L0.frame_dev && L0.spp != 1) return lt_fail(ctx, LT_ERR_INVALID_ARG, "a captured frame renders one frame");
    const size_t n = (size_t)L0.width * L0.height;
    // frames per launch: what the sample buffer holds, and items that fit 32 bits
    const size_t items = (size_t)((L0.width + 7) / 8) * ((L0.height + 7) / 8) * 64;
    uint32_t group = (uint32_t)std::max<size_t>(
        1, std::min<size_t>({L0.spp, kPathSampleBytes / (n * sizeof(float4)), (1ull << 31) / items}));
    if (group > 1 && ps.capacity < group * n) {
        path_samples_free(ps);
        if (hipMalloc(&ps.rad, group * n * sizeof(float4)) == hipSuccess) {
            ps.capacity = group * n;
        } else {  // no room: frame by frame, which needs no buffer
            (void)hipGetLastError();
            ps.rad = nullptr;
            group = 1;
        }
    }
    SceneView sv = make_scene_view(ctx);
    auto* cnt = (unsigned long long*)d_counts;
    if (count) hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, ctx->stream, (uint32_t*)d_counts, 2u * kCountSlots);
    phase_mark(ctx);
    for (uint32_t f = 0; f < L0.spp; f += group) {
        PathLaunch L = L0;
        L.frame_start = L0.frame_start + f;
        L.spp = std::min(group, L0.spp - f);
        L.regen_min = ctx->tuning.regen_min ? ctx->tuning.regen_min : 4u;
        const uint32_t grid = work_blocks(items * L.spp, (uint32_t)blocks, kTraceBlock / 64);
        if (work_counted(items * L.spp, grid, kTraceBlock / 64, true))
            hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, ctx->stream, ctx->counters, 1u);
        if (count)
            hipLaunchKernelGGL((k_path_regen<true>), dim3(grid), dim3(kTraceBlock), 0, ctx->stream, sv, L, accum,
                               ps.rad, ctx->counters, ctx->spill, cnt);
        else
            hipLaunchKernelGGL((k_path_regen<false>), dim3(grid), dim3(kTraceBlock), 0, ctx->stream, sv, L, accum,
                               ps.rad, ctx->counters, ctx->spill, cnt);
        if (L.spp > 1u)
            hipLaunchKernelGGL(k_path_mean, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, ps.rad, accum,
                               (uint32_t)n, L.frame_start, L.spp);
    }
    LT_HIP(ctx, hipGetLastError());
    return LT_OK;
}
