// adjoint.hip — the differentiable Path estimator and its path-replay
// adjoint on gfx950.
//
// No reference counterpart (the reference renders but does not
// differentiate).  The estimator is the Path kernel's per-sample logic
// (src/shaders/integrators/path/path.rgen:26-104, pt_commons.glsl:3-42)
// without roulette; the albedo and roughness textures aid / rid are read
// from per-variant texel arrays.  Derivatives hold the random numbers fixed
// and sampling detached (directions, lobe choices, pdfs and MIS weights are
// constants): path-replay backpropagation (Vicini, Speierer and Jakob 2021)
// adds, at vertex j of a replayed sample with radiance L and adjoint delta,
//   delta . (df_j / f_j) (L - radiance gathered before j's continuation)
// for the sampled continuation and delta . T_j dN_j for the next-event
// terms, scattered to the four texels of the bilinear footprint with float
// atomics.  The first pass's L comes from the forward's per-sample cache
// (one 12-B record per sample in HBM) or is recomputed.
//
// Texel derivatives: Lambertian albedo, and the principled BSDF with
// metallic, spec_trans, specular_tint, clearcoat, flatness and anisotropy
// zero (GGX reflection + Disney diffuse), alpha = max(0.001, r^2):
//   f = S(alpha) + albedo g(r) / pi,  dS/dr = S (dlnD/dalpha + dlnG/dalpha) 2r
//   dlnD/dalpha = -2/alpha + 4e/(alpha (1 + e)),  e = tan^2(h) c_h / alpha^2
//   dlnG/dalpha = -G (dL(wo) + dL(wi)),  dL = alpha c tan^2 / (2 sqrt(1 + c alpha^2 tan^2))
//   g = (1 - f_i/2)(1 - f_o/2) + rr (f_i + f_o^2 f_i (rr - 1)),  rr = 2 r^2 cos_i^2
// (c = the clamped azimuth factor of the Smith / GGX formulas; a lobe with
// alpha <= 0.0064 is the reference's delta reflection and has no roughness
// derivative).
#include <hip/hip_runtime.h>

#include "adjoint.h"
#include "context.h"
#include "dev_scene.h"
// The adjoint kernels test each hit leaf before taking another node: their
// traversals run beside a long per-lane replay state, and the leaf queue's
// deferred culling cost them more node steps than it saved in idle lanes.
#define LT_NODE_PEND_MAX 0
#include "dev_count.h"
#include "dev_trace.h"

using namespace ltd;

namespace {

constexpr float ADJ_TMIN = 0.001f;    // path.rgen:19
constexpr float ADJ_TMAX = 10000.0f;  // path.rgen:20

// bilinear footprint (repeat addressing, texel centres at (i + 0.5) / size)
struct Taps {
    uint32_t i00, i01, i10, i11;
    float ax, ay;
};

LT_DEV Taps taps_of(int W, int H, f2 uv) {
    float fx = uv.x * (float)W - 0.5f, fy = uv.y * (float)H - 0.5f;
    float x0f = floorf(fx), y0f = floorf(fy);
    Taps t;
    t.ax = fx - x0f;
    t.ay = fy - y0f;
    int x0 = ((int)x0f % W + W) % W, y0 = ((int)y0f % H + H) % H;
    int x1 = (x0 + 1) % W, y1 = (y0 + 1) % H;
    t.i00 = (uint32_t)(y0 * W + x0);
    t.i01 = (uint32_t)(y0 * W + x1);
    t.i10 = (uint32_t)(y1 * W + x0);
    t.i11 = (uint32_t)(y1 * W + x1);
    return t;
}

// d[texel * stride + c]
LT_DEV float fetch(const float* __restrict__ d, size_t stride, size_t c, const Taps& t) {
    const float top = d[stride * t.i00 + c] * (1.0f - t.ax) + d[stride * t.i01 + c] * t.ax;
    const float bot = d[stride * t.i10 + c] * (1.0f - t.ax) + d[stride * t.i11 + c] * t.ax;
    return top * (1.0f - t.ay) + bot * t.ay;
}

struct DMat {
    Mat m;
    f3 amult;  // the material's albedo factor
    Taps ta, tr;
    bool ta_on, tr_on;
};

// load_material (bsdf_commons.glsl:16-22) with the variant's texels
LT_DEV DMat load_dmat(const SceneView& sv, const AdjLaunch& L, const float* alb, const float* rgh, uint32_t idx,
                      f2 uv) {
    DMat d;
    uint32_t* dst = (uint32_t*)&d.m;
    const uint32_t* s32 = (const uint32_t*)(sv.mats + idx);
#pragma unroll
    for (int i = 0; i < 26; i++) dst[i] = s32[i];
    d.amult = d.m.albedo;
    d.ta_on = d.tr_on = false;
    if (d.m.texture_id > -1) {
        if (alb && d.m.texture_id == L.aid) {
            d.ta = taps_of((int)L.aw, (int)L.ah, uv);
            d.ta_on = true;
            d.m.albedo = d.amult * mk3(fetch(alb, 3u * L.texel_step, 0u, d.ta), fetch(alb, 3u * L.texel_step, L.texel_step, d.ta),
                                      fetch(alb, 3u * L.texel_step, 2u * L.texel_step, d.ta));
        } else {
            const float4 t = tex_bilinear(sv, d.m.texture_id, uv);
            d.m.albedo = d.m.albedo * mk3(t.x, t.y, t.z);
        }
    }
    if (sv.rough) {
        const int rt = sv.rough[idx];
        if (rt > -1) {
            if (rgh && rt == L.rid) {
                d.tr = taps_of((int)L.rw, (int)L.rh, uv);
                d.tr_on = true;
                d.m.roughness = fetch(rgh, L.texel_step, 0u, d.tr);
            } else {
                d.m.roughness = tex_bilinear(sv, rt, uv).x;
            }
        }
    }
    return d;
}

// ---- BSDF derivatives (local frame) ----
LT_DEV void diffuse_g(f3 wo, f3 wi, float r, float& g, float& dg) {
    const f3 h = normalize(wi + wo);
    const float wh = dot(wo, h);
    const float fd90 = 0.5f + 2.0f * wh * wh * r, dfd90 = 2.0f * wh * wh;
    const float Pi = pow5m(wi.z), Po = pow5m(wo.z);
    const float fi = 1.0f + (fd90 - 1.0f) * Pi, fo = 1.0f + (fd90 - 1.0f) * Po;
    const float dfi = dfd90 * Pi, dfo = dfd90 * Po;
    const float rr = 2.0f * (r * r) * wi.z * wi.z, drr = 4.0f * r * wi.z * wi.z;
    const float inner = fi + fo * fi * fo * (rr - 1.0f);
    g = (1.0f - 0.5f * fi) * (1.0f - 0.5f * fo) + rr * inner;
    const float dinner = dfi + (2.0f * fo * dfo * fi + fo * fo * dfi) * (rr - 1.0f) + fo * fo * fi * drr;
    dg = -0.5f * dfi * (1.0f - 0.5f * fo) - 0.5f * dfo * (1.0f - 0.5f * fi) + drr * inner + rr * dinner;
}

LT_DEV bool tan2_c(f3 w, float& t2, float& c) {
    const float c2 = w.z * w.z;
    const float s2 = fmaxf(1.0f - c2, 0.0f);
    t2 = s2 / c2;
    if (isinf(t2)) return false;
    c = s2 == 0.0f ? 1.0f : (clampf(w.x * w.x, 0.0f, 1.0f) + clampf(w.y * w.y, 0.0f, 1.0f)) / s2;
    return true;
}

LT_DEV float spec_dlog_dr(f3 wo, f3 wi, float r) {
    const float alpha = fmaxf(0.001f, r * r);
    if (alpha <= 0.0064f) return 0.0f;
    const f3 h = normalize(wo + wi);
    float t2, c, dlnD = 0.0f;
    if (tan2_c(h, t2, c)) {
        const float e = t2 * c / (alpha * alpha);
        dlnD = -2.0f / alpha + 4.0f * e / (alpha * (1.0f + e));
    }
    float Ls = 0.0f, dLs = 0.0f;
    if (tan2_c(wo, t2, c)) {
        const float q = sqrtf(1.0f + c * alpha * alpha * t2);
        Ls += 0.5f * (q - 1.0f);
        dLs += alpha * c * t2 / (2.0f * q);
    }
    if (tan2_c(wi, t2, c)) {
        const float q = sqrtf(1.0f + c * alpha * alpha * t2);
        Ls += 0.5f * (q - 1.0f);
        dLs += alpha * c * t2 / (2.0f * q);
    }
    const float G = 1.0f / (1.0f + Ls);
    return (dlnD - G * dLs) * (2.0f * r);
}

struct DF {
    f3 f, dfa, dfr;
};

// eval_bsdf plus texel derivatives
LT_DEV DF eval_d(const DMat& d, f3 n_s, f3 wo_w, f3 wi_w, bool side, float& pdf) {
    DF o;
    float pr;
    o.f = eval_bsdf(n_s, wo_w, d.m, side, wi_w, pdf, pr, false);
    o.dfa = o.dfr = mk3(0.0f);
    if (!(d.ta_on || d.tr_on)) return o;
    f3 T, B;
    branchless_onb(n_s, T, B);
    const f3 wo = to_local(wo_w, T, B, n_s), wi = to_local(wi_w, T, B, n_s);
    if (d.m.bsdf_type == LT_BSDF_DIFFUSE) {
        if (fminf(wi.z, wo.z) > 0.0f) o.dfa = mk3(INV_PI);
        return o;
    }
    if (d.m.bsdf_type != LT_BSDF_PRINCIPLED) return o;
    float ps, pd, pc, pt;
    init_probs(d.m, fresnel_dielectric(wo.z, d.m.ior, side), side, ps, pd, pc, pt);
    f3 diff = mk3(0.0f);
    if (fminf(wi.z, wo.z) > 0.0f && pd > 0.0f) {
        float g, dg;
        diffuse_g(wo, wi, d.m.roughness, g, dg);
        diff = d.m.albedo * g * INV_PI;
        o.dfa = mk3(g * INV_PI);
        o.dfr = d.m.albedo * dg * INV_PI;
    }
    if (ps > 0.0f && !(wo.z * wi.z < 0.0f) && wo.z != 0.0f && wi.z != 0.0f)
        o.dfr += (o.f - diff) * spec_dlog_dr(wo, wi, d.m.roughness);
    return o;
}

// sample_bsdf plus derivatives of the sampled lobe's value
LT_DEV DF sample_d(const DMat& d, f3 n_s, f3 wo_w, bool side, f3& wi_w, float& pdf, float& cos_t, float r0,
                   float r1, float r2) {
    DF o;
    o.f = sample_bsdf(n_s, wo_w, d.m, 1, side, wi_w, pdf, cos_t, r0, r1, r2);
    o.dfa = o.dfr = mk3(0.0f);
    if (!(d.ta_on || d.tr_on)) return o;
    f3 T, B;
    branchless_onb(n_s, T, B);
    const f3 wo = to_local(wo_w, T, B, n_s), wi = to_local(wi_w, T, B, n_s);
    if (d.m.bsdf_type == LT_BSDF_DIFFUSE) {
        if (fminf(wi.z, wo.z) > 0.0f) o.dfa = mk3(INV_PI);
        return o;
    }
    if (d.m.bsdf_type != LT_BSDF_PRINCIPLED || wo.z <= 0.0f) return o;
    float ps, pd, pc, pt;
    init_probs(d.m, fresnel_dielectric(wo.z, d.m.ior, side), side, ps, pd, pc, pt);
    if (r2 < ps) {
        o.dfr = o.f * spec_dlog_dr(wo, wi, d.m.roughness);
    } else if (r2 > ps + pc && r2 <= ps + pc + pd) {
        if (fminf(wi.z, wo.z) > 0.0f) {
            float g, dg;
            diffuse_g(wo, wi, d.m.roughness, g, dg);
            o.dfa = mk3(g * INV_PI);
            o.dfr = d.m.albedo * dg * INV_PI;
        }
    }
    return o;
}

LT_DEV bool nz(f3 a) { return a.x != 0.0f || a.y != 0.0f || a.z != 0.0f; }

// one vertex's texel gradients: qa per albedo channel, qr for roughness
LT_DEV void scatter(const AdjLaunch& L, const DMat& d, float* __restrict__ ga, float* __restrict__ gr, f3 qa, float qr) {
    if (d.ta_on && nz(qa)) {
        const f3 q = qa * d.amult;
        const float w[4] = {(1.0f - d.ta.ax) * (1.0f - d.ta.ay), d.ta.ax * (1.0f - d.ta.ay),
                            (1.0f - d.ta.ax) * d.ta.ay, d.ta.ax * d.ta.ay};
        const uint32_t idx[4] = {d.ta.i00, d.ta.i01, d.ta.i10, d.ta.i11};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            float* g = ga + 3u * L.texel_step * idx[k];
            atomicAdd(g, w[k] * q.x);
            atomicAdd(g + L.texel_step, w[k] * q.y);
            atomicAdd(g + 2u * L.texel_step, w[k] * q.z);
        }
    }
    if (d.tr_on && qr != 0.0f) {
        const float w[4] = {(1.0f - d.tr.ax) * (1.0f - d.tr.ay), d.tr.ax * (1.0f - d.tr.ay),
                            (1.0f - d.tr.ax) * d.tr.ay, d.tr.ax * d.tr.ay};
        const uint32_t idx[4] = {d.tr.i00, d.tr.i01, d.tr.i10, d.tr.i11};
#pragma unroll
        for (int k = 0; k < 4; k++) atomicAdd(gr + L.texel_step * idx[k], w[k] * qr);
    }
}

LT_DEV f3 safe_inv(f3 f) {
    return {f.x != 0.0f ? 1.0f / f.x : 0.0f, f.y != 0.0f ? 1.0f / f.y : 0.0f, f.z != 0.0f ? 1.0f / f.z : 0.0f};
}

// A hit as the sample cache records it: instance, primitive, barycentrics
// (instance ~0: a miss), enough to rebuild the payload without a trace.  A
// record naming no point of a triangle of the scene (a miss, or a cache that
// no forward of this scene wrote) decodes as a miss, so any cache contents
// stay in bounds and give finite hit points.
LT_DEV void payload_from_record(const SceneView& sv, uint4 r, Payload& pl) {
    const float u = __uint_as_float(r.z), v = __uint_as_float(r.w);
    if (r.x >= sv.num_prims || r.y >= sv.tri_start[r.x + 1] - sv.tri_start[r.x] ||
        !(u >= -1e-3f && v >= -1e-3f && u + v <= 1.001f))
        pl.valid = false;  // ray.rmiss:13 — the other fields keep the last hit
    else
        fill_payload(sv, r.x, r.y, u, v, pl);
}

// the payload of a hit record that this scene's trace made
LT_DEV void payload_of(const SceneView& sv, uint4 r, Payload& pl) {
    if (r.x != 0xFFFFFFFFu)
        fill_payload(sv, r.x, r.y, __uint_as_float(r.z), __uint_as_float(r.w), pl);
    else
        pl.valid = false;  // ray.rmiss:13 — the other fields keep the last hit
}

template <bool COUNT>
LT_DEV void closest(const SceneView& sv, f3 o, f3 d, const TraceStack& stk, Payload& pl, Ctr& c, uint4* rec) {
    HitRec h;
    if (COUNT) c.closest++;
    const bool hit = trace_bvh<false, COUNT>(sv, o, d, ADJ_TMIN, ADJ_TMAX, h, stk, c.nodes, c.tris);
    *rec = hit ? make_uint4(h.inst, h.prim, __float_as_uint(h.u), __float_as_uint(h.v))
               : make_uint4(0xFFFFFFFFu, 0u, 0u, 0u);
    payload_of(sv, *rec, pl);
}

// The path records of one sample in the sample cache: hit records
// [k][bounce][2][item] (the path's closest hit, the NEE MIS ray's hit), a flag
// word [k][item] with 3 bits per bounce (NEE occlusion traced, occluded, MIS
// ray traced).  The forward writes them; the replay reads them instead of
// tracing, and traces what the forward did not (a light whose contribution
// was zero but whose derivative is not).
struct AdjRec {
    uint4* hits;  // nullptr: no records
    uint32_t* flags;
    size_t n;     // items
    uint32_t depth, k, i;
    LT_DEV uint4* hit(int bounce, int plane) const {
        return hits + (((size_t)k * depth + (size_t)bounce) * 2u + (size_t)plane) * n + i;
    }
};

// The rays of a sample that its variants share.  The 32 (say) variants of a
// pixel differ in the texels of one or two textures, the random numbers are
// the same, so their paths coincide until a texel changes a sampled direction
// (a glossy lobe's roughness): most of them to the end.  A wave holds the
// variants of few pixels, and stepping their few distinct rays costs as much
// as 64 different ones.  So it first walks each (pixel, sample) of a run of
// groups once, a lane each, with the first variant's texels, and keeps its
// rays and hits here; then the variants run sample by sample and take a hit
// from here where their own ray is bit for bit the same, and trace where it is
// not.  At 512x512, 32 variants, 8 samples, depth 6: BVH8 nodes 1.77 G ->
// 0.31 G, VALU instructions 18.7 G -> 12.4 G, forward 32.4 -> 27.8 ms (one
// group per walk, 16 of its 64 lanes in use: 15.4 G and 35.7 ms).  What is
// left is shading, and the rays of glossy lobes that leave the shared ones
// (31 of 64 lanes active).
//   per bounce: hit record; ray direction and tag; MIS hit record; MIS
//   direction.  Tag: random numbers drawn before the bounce * 8 + flags
//   (1 shadow ray traced, 2 occluded, 4 MIS ray traced)
// The same draws, the same hits before and the same direction make the same
// origin, shadow ray and MIS origin: nothing else of a ray comes from a texel.
struct AdjTrunk {
    uint4* base;     // the wave's: [bounce][4][64]; nullptr: no sharing
    uint32_t slot;   // this lane's (pixel, sample)
    uint32_t depth;  // bounces kept
    bool write;      // wave-uniform: the walk that fills it
    static constexpr uint32_t kEnd = 0xFFFFFFFFu;  // tag: the walk ended before this bounce
    LT_DEV uint4* at(int bounce, int f) const { return base + ((size_t)bounce * 4u + (size_t)f) * 64u + slot; }
};

LT_DEV bool same_bits(uint4 r, f3 d) {
    return r.x == __float_as_uint(d.x) && r.y == __float_as_uint(d.y) && r.z == __float_as_uint(d.z);
}

template <bool COUNT>
LT_DEV bool occluded(const SceneView& sv, f3 o, f3 d, float tmax, const TraceStack& stk, Ctr& c) {
    HitRec h;
    if (COUNT) c.shadow++;
    return trace_bvh<true, COUNT>(sv, o, d, 0.0f, tmax, h, stk, c.snodes, c.stris);
}

// One sample of pixel (x, y).  REPLAY: the same path again with its radiance
// Lt and adjoint radiance delta, scattering texel gradients into ga / gr.
// TRUNK: with shared rays (T).
template <bool REPLAY, bool COUNT, bool TRUNK>
LT_DEV f3 adj_sample(const SceneView& sv, const AdjLaunch& L, const float* alb, const float* rgh, uint32_t x,
                     uint32_t y, uint32_t word, f3 Lt, f3 delta, float* ga, float* gr, const TraceStack& stk,
                     Ctr& cnt, const AdjRec& R, const AdjTrunk& T) {
    bool shared = TRUNK && T.base != nullptr;  // every ray so far was the shared one
    const bool rec_on = R.hits != nullptr;
    uint32_t fl_word = (REPLAY && rec_on) ? R.flags[(size_t)R.k * R.n + R.i] : 0u;
    RNG seed = {x, y, word, 0u};
    const float r0 = rnd(seed);
    const float r1 = rnd(seed);
    const float ux = ((float)x + 0.5f + (r0 - 0.5f)) / (float)L.width;
    const float uy = ((float)y + 0.5f + (r1 - 0.5f)) / (float)L.height;
    const f4 o4 = mul4(L.inv_view, f4{0.0f, 0.0f, 0.0f, 1.0f});
    const f4 tg = mul4(L.inv_projection, f4{ux * 2.0f - 1.0f, uy * 2.0f - 1.0f, 1.0f, 1.0f});
    const f3 tn = normalize(mk3(tg.x, tg.y, tg.z));
    const f4 d4 = mul4(L.inv_view, f4{tn.x, tn.y, tn.z, 0.0f});
    f3 origin = {o4.x, o4.y, o4.z};
    f3 direction = {d4.x, d4.y, d4.z};
    f3 col = mk3(0.0f), thr = mk3(1.0f);
    bool last_specular = false;
    Payload pl;
    pl.valid = false;
    pl.triangle_idx = pl.instance_idx = 0xFFFFFFFFu;
    pl.pos = pl.n_s = pl.n_g = mk3(0.0f);
    const float pick = 1.0f / (float)sv.total_light_triangle_cnt;
    int depth = 0;
    for (;; depth++) {
        uint32_t t_flags = 0u;  // of this bounce's shared rays
        const uint32_t tag = seed.w << 3;
        if (TRUNK) shared = shared && depth < (int)T.depth;
        if (REPLAY && rec_on) {
            payload_from_record(sv, *R.hit(depth, 0), pl);
        } else {
            uint4 r;
            bool have = false;
            if (TRUNK && shared && !T.write) {
                const uint4 d = *T.at(depth, 1);
                shared = have = same_bits(d, direction) && (d.w & ~7u) == tag;
                t_flags = have ? d.w & 7u : 0u;
            }
            if (have) {
                r = *T.at(depth, 0);
                payload_of(sv, r, pl);
                if (COUNT) cnt.closest++;
            } else {
                closest<COUNT>(sv, origin, direction, stk, pl, cnt, &r);
            }
            if (rec_on) *R.hit(depth, 0) = r;
            if (TRUNK && shared && T.write) {
                *T.at(depth, 0) = r;
                *T.at(depth, 1) = make_uint4(__float_as_uint(direction.x), __float_as_uint(direction.y),
                                             __float_as_uint(direction.z), tag);
            }
        }
        if (!pl.valid) {
            col += thr * ld3(L.sky_col);
            break;
        }
        const Payload hp = pl;
        const DMat dm = load_dmat(sv, L, alb, rgh, hp.material_idx, hp.uv);
        if (depth == 0 || last_specular) col += thr * dm.m.emissive;
        if (depth >= L.max_depth - 1) break;
        const f3 wo = -direction;
        f3 n_s = hp.n_s, n_g = hp.n_g;
        bool side = true;
        if (dot(hp.n_g, wo) < 0.0f) n_g = -n_g;
        if (dot(n_g, hp.n_s) < 0.0f) {
            n_s = -n_s;
            side = false;
        }
        origin = offset_ray(hp.pos, n_g);
        last_specular = is_specular(dm.m);
        f3 qa = mk3(0.0f);
        float qr = 0.0f;
        if (!last_specular) {  // pt_commons.glsl:3-42 / pick pdf (path.rgen:76)
            f4 r4;
            r4.x = rnd(seed);
            r4.y = rnd(seed);
            r4.z = rnd(seed);
            r4.w = rnd(seed);
            f3 wi;
            float wi_len, pw, pa, cfl;
            LightRecord rec;
            rec.triangle_idx = 0;
            rec.instance_idx = 0;
            const f3 Le = sample_light_Li(sv, r4, hp.pos, pw, wi, wi_len, pa, cfl, rec);
            const f3 pp = offset_ray2(hp.pos, n_s);
            const float cos_x = dot(n_s, wi);
            f3 res = mk3(0.0f);
            float bpdf;
            if (REPLAY) {
                const DF fl = eval_d(dm, n_s, wo, wi, side, bpdf);
                if (pw > 0.0f) {
                    const float mis = (rec.flags & LT_LIGHT_DELTA) ? 1.0f : 1.0f / (1.0f + bpdf / pw);
                    const f3 ka = mis * fabsf(cos_x) * Le / pw;
                    const f3 contrib = mis * fl.f * fabsf(cos_x) * Le / pw;
                    bool occ = false;
                    if (nz(contrib) || nz(fl.dfa) || nz(fl.dfr)) {
                        const uint32_t b = fl_word >> (3 * depth);
                        occ = (rec_on && (b & 1u)) ? (b & 2u) != 0u : occluded<COUNT>(sv, pp, wi, wi_len - EPS, stk, cnt);
                    }
                    if ((nz(contrib) || nz(fl.dfa) || nz(fl.dfr)) && !occ) {
                        res += contrib;
                        const f3 w = delta * thr / pick * ka;
                        qa += w * fl.dfa;
                        qr += dot(w, fl.dfr);
                    }
                }
            } else {
                float brev;
                const f3 f = eval_bsdf(n_s, wo, dm.m, side, wi, bpdf, brev, false);
                if (pw > 0.0f) {
                    const float mis = (rec.flags & LT_LIGHT_DELTA) ? 1.0f : 1.0f / (1.0f + bpdf / pw);
                    const f3 contrib = mis * f * fabsf(cos_x) * Le / pw;
                    if (nz(contrib)) {
                        bool occ;
                        if (TRUNK && (t_flags & 1u) && !T.write) {
                            occ = (t_flags & 2u) != 0u;
                            if (COUNT) cnt.shadow++;
                        } else {
                            occ = occluded<COUNT>(sv, pp, wi, wi_len - EPS, stk, cnt);
                        }
                        if (TRUNK && T.write) t_flags |= occ ? 3u : 1u;
                        fl_word |= (occ ? 3u : 1u) << (3 * depth);
                        if (!occ) res += contrib;
                    }
                }
            }
            if ((rec.flags & 7u) == LT_LIGHT_AREA) {
                const float s0 = rnd(seed), s1 = rnd(seed), s2 = rnd(seed);
                float bp, cx;
                f3 wb;
                const DF fb = REPLAY ? sample_d(dm, n_s, wo, side, wb, bp, cx, s0, s1, s2)
                                     : DF{sample_bsdf(n_s, wo, dm.m, 1, side, wb, bp, cx, s0, s1, s2), mk3(0.0f),
                                          mk3(0.0f)};
                if (bp != 0.0f) {
                    if (REPLAY && rec_on && ((fl_word >> (3 * depth)) & 4u)) {
                        payload_from_record(sv, *R.hit(depth, 1), pl);
                    } else if (TRUNK && (t_flags & 4u) && !T.write && same_bits(*T.at(depth, 3), wb)) {
                        const uint4 r = *T.at(depth, 2);
                        payload_of(sv, r, pl);
                        if (COUNT) cnt.closest++;
                        if (rec_on) *R.hit(depth, 1) = r;
                        fl_word |= 4u << (3 * depth);
                    } else {
                        uint4 r;
                        closest<COUNT>(sv, pp, wb, stk, pl, cnt, &r);
                        if (!REPLAY && rec_on) *R.hit(depth, 1) = r;
                        if (!REPLAY) fl_word |= 4u << (3 * depth);
                        if (TRUNK && shared && T.write) {
                            t_flags |= 4u;
                            *T.at(depth, 2) = r;
                            *T.at(depth, 3) = make_uint4(__float_as_uint(wb.x), __float_as_uint(wb.y),
                                                         __float_as_uint(wb.z), 0u);
                        }
                    }
                    if (pl.triangle_idx == rec.triangle_idx && pl.instance_idx == rec.instance_idx) {
                        const float wl = length(pl.pos - hp.pos);
                        const float gg = fabsf(dot(pl.n_s, -wb)) / (wl * wl);
                        const float mis = 1.0f / (1.0f + pa / (gg * bp));
                        res += fb.f * mis * fabsf(cx) * Le / bp;
                        if (REPLAY) {
                            const f3 w = delta * thr / pick * (mis * fabsf(cx) * Le / bp);
                            qa += w * fb.dfa;
                            qr += dot(w, fb.dfr);
                        }
                    }
                }
            }
            col += thr * res / pick;
            if (TRUNK && shared && T.write) T.at(depth, 1)->w = tag | t_flags;
        }
        const float s0 = rnd(seed), s1 = rnd(seed), s2 = rnd(seed);
        float pdf, cos_t;
        if (REPLAY) {
            const DF fc = sample_d(dm, n_s, wo, side, direction, pdf, cos_t, s0, s1, s2);
            if (pdf != 0.0f) {
                const f3 w = delta * (Lt - col) * safe_inv(fc.f);
                qa += w * fc.dfa;
                qr += dot(w, fc.dfr);
            }
            scatter(L, dm, ga, gr, qa, qr);
            if (pdf == 0.0f) break;
            thr *= fc.f * fabsf(cos_t) / pdf;
        } else {
            const f3 f = sample_bsdf(n_s, wo, dm.m, 1, side, direction, pdf, cos_t, s0, s1, s2);
            if (pdf == 0.0f) break;
            thr *= f * fabsf(cos_t) / pdf;
        }
    }
    // a variant may go on where the walk could not
    if (TRUNK && T.write && shared && depth + 1 < (int)T.depth) T.at(depth + 1, 1)->w = AdjTrunk::kEnd;
    if (!REPLAY && rec_on) R.flags[(size_t)R.k * R.n + R.i] = fl_word;
    return col;
}

// Three waves per SIMD (168 VGPRs): about as fast as four on the
// differentiable Cornell box and ~20 % faster than the unconstrained two.
// Four (128 VGPRs, 304-444 B of scratch per lane) gave wrong gradients in the
// replay test once the BVH8 internal children moved to the low slots, with
// no cause found in this source, so it is not used.
#ifndef LT_ADJ_WAVES
#define LT_ADJ_WAVES 3
#endif
// COUNT: the counting variant (rays traced, BVH8 nodes and triangles visited,
// summed into counts)
template <bool BACKWARD, bool COUNT>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(LT_ADJ_WAVES))) void k_adjoint(SceneView sv, AdjLaunch L, AdjBuffers B,
                                                         uint32_t* __restrict__ work, uint32_t* __restrict__ spill,
                                                         uint4* trunk,
                                                         unsigned long long* __restrict__ counts) {
    Ctr cnt{0u, 0u, 0u, 0u, 0u, 0u};
    __shared__ uint32_t s_stack[ltb::kLdsWords * kTraceBlock];
    const uint32_t gtid = blockIdx.x * blockDim.x + threadIdx.x;
    const TraceStack stk{s_stack + threadIdx.x, spill + (size_t)gtid * (ltb::kStackTotal - ltb::kLdsStack)};
    const uint32_t lane = threadIdx.x & 63u;
    // from one variant's texels to the next one's
    const size_t na = L.texel_step != 1u ? 1u : 3u * (size_t)L.aw * L.ah;
    const size_t nr = L.texel_step != 1u ? 1u : (size_t)L.rw * L.rh;
    const size_t npx = (size_t)L.width * L.height;
    const float inv_spp = 1.0f / (float)L.spp;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(gtid >> 6));
    AdjTrunk T{nullptr, 0u, L.trunk_depth, false};
    if (!BACKWARD && L.trunk_depth) T.base = trunk + (size_t)wave * L.trunk_depth * 4u * 64u;
    // n_items is a multiple of 64; a tile of the wave is a run of up to L.run
    // groups of 64 items
    const uint32_t n_groups = L.n_items >> 6, run = BACKWARD ? 1u : L.run;
    WaveTiles wt = wave_tiles((n_groups + run - 1u) / run * 64u, work, true);
    while (next_tile(wt)) {
        const uint32_t g0 = (wt.base >> 6) * run, ng = min(run, n_groups - g0);
        uint32_t i = g0 * 64u + lane;
        uint32_t v, p, x, y;
        bool inside;
        const float *alb, *rgh;
        size_t pix;
        auto set_item = [&]() {
            v = i % L.variants;
            p = i / L.variants;
            const uint32_t tile = p >> 6, w = p & 63u;
            x = (tile % L.tiles_x) * 8 + (w & 7u);
            y = (tile / L.tiles_x) * 8 + (w >> 3);
            inside = x < L.width && y < L.height;
            alb = L.aid >= 0 ? B.albedo + na * v : nullptr;
            rgh = L.rid >= 0 ? B.rough + nr * v : nullptr;
            pix = npx * v + (size_t)y * L.width + x;
        };
        set_item();
        if (BACKWARD && !inside) continue;
        // the sample cache's path records of sample k of this item (none
        // without a cache or beyond kAdjRecMaxDepth bounces)
        auto rec_of = [&](uint32_t k) {
            if (!B.cache || L.rec_depth == 0u) return AdjRec{nullptr, nullptr, 0, 0, 0, 0};
            uint4* hits = reinterpret_cast<uint4*>(B.cache + (size_t)L.spp * 3u * L.n_items);
            uint32_t* flags = reinterpret_cast<uint32_t*>(hits + (size_t)L.spp * L.rec_depth * 2u * L.n_items);
            return AdjRec{hits, flags, (size_t)L.n_items, L.rec_depth, k, i};
        };
        if (!BACKWARD) {
            f3 sum = mk3(0.0f);
            // a batch: the samples whose (pixel, sample) pairs fill the wave
            // (all of them if the run has more than one group)
            const uint32_t p0 = g0 * 64u / L.variants, np = ((g0 + ng) * 64u - 1u) / L.variants - p0 + 1u;
            const uint32_t batch = T.base ? min(L.spp, max(1u, 64u / np)) : L.spp;
            for (uint32_t k0 = 0; k0 < L.spp; k0 += batch) {
                const uint32_t kn = min(batch, L.spp - k0);
                // step 0 walks the shared rays, the others run the batch's
                // samples of group g, one after another
                uint32_t g = 0u, k = 0u;
                T.write = T.base != nullptr;
                for (;;) {
                    uint32_t sx = x, sy = y, word = k0 + k;
                    const float *sa = alb, *sr = rgh;
                    bool go = inside;
                    T.slot = (p - p0) * batch + k;
                    if (T.write) {
                        const uint32_t j = lane / batch, q = p0 + j, qt = q >> 6;
                        sx = (qt % L.tiles_x) * 8 + (q & 7u);
                        sy = (qt / L.tiles_x) * 8 + ((q & 63u) >> 3);
                        word = k0 + lane % batch;
                        go = j < np && lane % batch < kn && sx < L.width && sy < L.height;
                        sa = L.aid >= 0 ? B.albedo : nullptr;
                        sr = L.rid >= 0 ? B.rough : nullptr;
                        T.slot = lane;
                    }
                    const Ctr before = cnt;
                    if (go) {
                        const AdjRec R = T.write ? AdjRec{nullptr, nullptr, 0, 0, 0, 0} : rec_of(word);
                        const f3 c = adj_sample<false, COUNT, true>(sv, L, sa, sr, sx, sy, word ^ L.seed, mk3(0.0f),
                                                                    mk3(0.0f), nullptr, nullptr, stk, cnt, R, T);
                        if (!T.write) {
                            if (B.cache) {
                                float* cp = B.cache + (size_t)word * 3 * L.n_items + i;
                                cp[0] = c.x;
                                cp[L.n_items] = c.y;
                                cp[2 * (size_t)L.n_items] = c.z;
                            }
                            if (!isnan(luminance(c))) sum += c;  // path.rgen:102-104
                        }
                    }
                    if (T.write) {
                        if (COUNT) {  // its rays are counted where the variants take them
                            cnt.closest = before.closest;
                            cnt.shadow = before.shadow;
                        }
                        T.write = false;
                        __threadfence_block();  // written before they are read
                        __builtin_amdgcn_wave_barrier();
                        continue;
                    }
                    if (++k < kn) continue;
                    k = 0u;
                    if (k0 + batch >= L.spp) {
                        if (inside) {
                            B.images[3 * pix + 0] = sum.x * inv_spp;
                            B.images[3 * pix + 1] = sum.y * inv_spp;
                            B.images[3 * pix + 2] = sum.z * inv_spp;
                        }
                        sum = mk3(0.0f);
                    }
                    if (++g == ng) break;
                    i += 64u;
                    set_item();
                }
                if (T.base) {  // read before the next batch's are written
                    __threadfence_block();
                    __builtin_amdgcn_wave_barrier();
                }
            }
        } else {
            const f3 delta = ld3(B.d_images + 3 * pix) * inv_spp;
            if (!nz(delta)) continue;
            float* ga = L.aid >= 0 ? B.g_albedo + na * v : nullptr;
            float* gr = L.rid >= 0 ? B.g_rough + nr * v : nullptr;
            for (uint32_t k = 0; k < L.spp; k++) {
                f3 c;
                if (B.cache) {
                    const float* cp = B.cache + (size_t)k * 3 * L.n_items + i;
                    c = mk3(cp[0], cp[L.n_items], cp[2 * (size_t)L.n_items]);
                } else {
                    c = adj_sample<false, COUNT, false>(sv, L, alb, rgh, x, y, k ^ L.seed, mk3(0.0f), mk3(0.0f), nullptr,
                                                        nullptr, stk, cnt, AdjRec{nullptr, nullptr, 0, 0, 0, 0}, T);
                }
                if (isnan(luminance(c))) continue;
                adj_sample<true, COUNT, false>(sv, L, alb, rgh, x, y, k ^ L.seed, c, delta, ga, gr, stk, cnt, rec_of(k), T);
            }
        }
    }
    if (COUNT) flush_counts(cnt, counts);
}

__global__ void k_fill_f32(float* __restrict__ p, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0.0f;
}

// out[c][r] = in[r][c] of a rows x cols matrix: the variants' texels
// interleaved, or their gradients taken apart again.  Bound by HBM.
constexpr uint32_t kTransTile = 64;
__global__ __launch_bounds__(256) void k_transpose(const float* __restrict__ in, size_t rows, size_t cols,
                                                   float* __restrict__ out) {
    __shared__ float s[kTransTile][kTransTile + 1];
    const size_t tc = (cols + kTransTile - 1) / kTransTile;
    const size_t r0 = blockIdx.x / tc * kTransTile, c0 = blockIdx.x % tc * kTransTile;
    const uint32_t lane = threadIdx.x & 63u, row = threadIdx.x >> 6;
    for (uint32_t j = row; j < kTransTile && r0 + j < rows; j += 4)
        if (c0 + lane < cols) s[j][lane] = in[(r0 + j) * cols + c0 + lane];
    __syncthreads();
    for (uint32_t j = row; j < kTransTile && c0 + j < cols; j += 4)
        if (r0 + lane < rows) out[(c0 + j) * rows + r0 + lane] = s[lane][j];
}

void transpose(const float* in, size_t rows, size_t cols, float* out, hipStream_t stream) {
    const size_t tiles = ((rows + kTransTile - 1) / kTransTile) * ((cols + kTransTile - 1) / kTransTile);
    hipLaunchKernelGGL(k_transpose, dim3((unsigned)tiles), dim3(256), 0, stream, in, rows, cols, out);
}

__global__ void k_zero_word(uint32_t* p) {
    if (threadIdx.x == 0) p[0] = 0u;
}

__global__ void k_zero_u64(unsigned long long* p, uint32_t n) {
    if (threadIdx.x < n) p[threadIdx.x] = 0ull;
}

}  // namespace

uint32_t adjoint_blocks(lt_context* ctx) {
    const uint32_t b = std::max(resident_blocks(reinterpret_cast<const void*>(&k_adjoint<false, false>), 0u),
                                resident_blocks(reinterpret_cast<const void*>(&k_adjoint<true, false>), 0u));
    return (uint32_t)ctx->num_cus * std::min(std::max(1u, ctx->tuning.path_blocks_per_cu), b);
}

lt_status launch_adjoint(lt_context* ctx, const AdjLaunch& launch, const AdjBuffers& buffers, bool backward,
                         const AdjWork& W, unsigned long long* counts, hipStream_t stream) {
    SceneView sv = make_scene_view(ctx);
    AdjLaunch L = launch;
    AdjBuffers B = buffers;
    const size_t V = L.variants, na = L.aid >= 0 ? (size_t)L.aw * L.ah * 3 : 0, nr = L.rid >= 0 ? (size_t)L.rw * L.rh : 0;
    if (!W.trunk) L.trunk_depth = 0u;
    L.texel_step = W.texels ? L.variants : 1u;
    if (W.texels) {  // [texel, channel][variant]
        float* t = W.texels;
        if (na) transpose(B.albedo, V, na, t, stream);
        if (nr) transpose(B.rough, V, nr, t + V * na, stream);
        B.albedo = t;
        B.rough = t + V * na;
        B.g_albedo = t + V * (na + nr);
        B.g_rough = B.g_albedo + V * na;
    }
    // The shared walk comes before the variants' own work in each wave, so it
    // pays where waves have several groups, and costs where a launch is one
    // round and its longest wave counts (256x200, 4 variants, 8 samples, 1.04
    // groups per wave: 4.1 ms without, 5.2 ms with).
    const uint32_t n_groups = L.n_items / 64u;
    if (n_groups / (W.blocks * (kTraceBlock / 64)) < kAdjTrunkMinGroups) L.trunk_depth = 0u;
    // groups per shared walk: as many as its 64 lanes hold all samples of,
    // while the waves keep a few runs each
    uint32_t run = 1u;
    if (!backward && L.trunk_depth) {
        auto pixels = [&](uint32_t g) {  // most pixels that a run of g groups meets
            return g * 64u % L.variants == 0u ? g * 64u / L.variants : (g * 64u - 2u) / L.variants + 2u;
        };
        while (run < 16u && (uint64_t)pixels(run + 1u) * L.spp <= 64u &&
               n_groups / (run + 1u) >= W.blocks * (kTraceBlock / 64) * 4u)
            run++;
        // lanes in use; 32 of 64 (512x512, 8 variants, 2 samples): 5.8 ms without, 5.9 ms with
        const uint64_t lanes = (uint64_t)pixels(run) * std::min<uint64_t>(L.spp, 64u / pixels(run));
        if (lanes < kAdjTrunkMinLanes) {
            L.trunk_depth = 0u;
            run = 1u;
        }
    }
    L.run = run;
    const uint32_t blocks = work_blocks((uint64_t)((n_groups + run - 1u) / run) * 64u, W.blocks, kTraceBlock / 64);
    hipLaunchKernelGGL(k_zero_word, dim3(1), dim3(64), 0, stream, W.work);
    if (counts) hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, stream, counts, (uint32_t)kCountSlots);
    if (backward) {
        auto fill = [&](float* p, size_t n) {
            hipLaunchKernelGGL(k_fill_f32, dim3((unsigned)std::min<size_t>((n + 255) / 256, 4096)), dim3(256), 0, stream, p,
                               n);
        };
        if (na) fill(B.g_albedo, V * na);
        if (nr) fill(B.g_rough, V * nr);
        if (counts)
            hipLaunchKernelGGL((k_adjoint<true, true>), dim3(blocks), dim3(kTraceBlock), 0, stream, sv, L, B, W.work,
                               W.spill, W.trunk, counts);
        else
            hipLaunchKernelGGL((k_adjoint<true, false>), dim3(blocks), dim3(kTraceBlock), 0, stream, sv, L, B, W.work,
                               W.spill, W.trunk, counts);
        if (W.texels) {
            if (na) transpose(B.g_albedo, na, V, buffers.g_albedo, stream);
            if (nr) transpose(B.g_rough, nr, V, buffers.g_rough, stream);
        }
    } else {
        if (counts)
            hipLaunchKernelGGL((k_adjoint<false, true>), dim3(blocks), dim3(kTraceBlock), 0, stream, sv, L, B, W.work,
                               W.spill, W.trunk, counts);
        else
            hipLaunchKernelGGL((k_adjoint<false, false>), dim3(blocks), dim3(kTraceBlock), 0, stream, sv, L, B, W.work,
                               W.spill, W.trunk, counts);
    }
    LT_HIP(ctx, hipGetLastError());
    return LT_OK;
}
