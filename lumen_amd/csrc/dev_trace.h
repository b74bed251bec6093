// dev_trace.h — BVH8 traversal for gfx950: closest hit and any hit.
//
// Semantics of the reference's queries (traceRayEXT with gl_RayFlagsOpaqueEXT,
// and TerminateOnFirstHit|SkipClosestHit for shadows;
// src/shaders/integrators/path/path.rgen:48, pt_commons.glsl:20-23):
//   closest = the triangle with the smallest t in [tmin, tmax], ties to the
//             smaller global triangle index;
//   any     = some triangle with t in [tmin, tmax].
// Triangle test: Woop, Benthin & Wald, JCGT 2013 (watertight, with the
// double-precision edge fallback), evaluated without fused multiply-adds so
// that t, u, v are bitwise those of the host restatement.
//
// Stack: a per-thread short stack in LDS (kLdsStack entries, stride = block
// size so a wave's accesses are bank-conflict free), continued in a global
// spill area (kStackTotal - kLdsStack entries per resident thread).
//
// What bounds it: VALU issue, at the few lanes of a wave that still traverse
// (node and triangle fetches are served by the caches).  The node step is
// therefore kept short: everything that depends on the ray alone (slab error
// bounds, cull margin) is set once per ray, the children's order comes from
// one axis of the node, and a node's hit leaves are queued as one entry
// (against per-node bounds, a nearest-child search and an entry per leaf:
// 2.07M bounce rays over the 1M-triangle terrain 733 -> 636 us, the 1080p Path
// frame 3.92 -> 3.56 ms).
#pragma once
#include "bvh_layout.h"
#include "context.h"
#include "dev_count.h"
#include "dev_math.h"
#include "dev_work.h"

namespace ltd {

struct RayPre {
    int kx, ky, kz;
    float Sx, Sy, Sz;
    f3 inv;
    f3 err;        // per axis: bound on the rounding of a slab distance
    float margin;  // bound on the rounding of a watertight t
};

LT_DEV float sel(f3 v, int k) { return k == 0 ? v.x : (k == 1 ? v.y : v.z); }

LT_DEV RayPre prep_ray(f3 d) {
#pragma clang fp contract(off)
    RayPre r;
    float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    int kz = (ax > ay) ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    int kx = kz + 1;
    if (kx == 3) kx = 0;
    int ky = kx + 1;
    if (ky == 3) ky = 0;
    float dz = sel(d, kz);
    if (dz < 0.0f) {
        int t = kx;
        kx = ky;
        ky = t;
    }
    r.kx = kx;
    r.ky = ky;
    r.kz = kz;
    r.Sx = sel(d, kx) / dz;
    r.Sy = sel(d, ky) / dz;
    r.Sz = 1.0f / dz;
    // box-test reciprocal; exact zeros get a tiny same-signed stand-in
    const float tiny = 1e-30f;
    r.inv = {1.0f / (fabsf(d.x) < tiny ? copysignf(tiny, d.x) : d.x),
             1.0f / (fabsf(d.y) < tiny ? copysignf(tiny, d.y) : d.y),
             1.0f / (fabsf(d.z) < tiny ? copysignf(tiny, d.z) : d.z)};
    return r;
}

// Woop et al. 2013, listing 1 (no back-face culling)
LT_DEV bool isect_tri(f3 A0, f3 B0, f3 C0, f3 o, const RayPre& rp, float tmin, float tmax, float& t_out,
                      float& u_out, float& v_out) {
#pragma clang fp contract(off)
    const f3 A = A0 - o, B = B0 - o, C = C0 - o;
    const float Akz = sel(A, rp.kz), Bkz = sel(B, rp.kz), Ckz = sel(C, rp.kz);
    const float Ax = sel(A, rp.kx) - rp.Sx * Akz, Ay = sel(A, rp.ky) - rp.Sy * Akz;
    const float Bx = sel(B, rp.kx) - rp.Sx * Bkz, By = sel(B, rp.ky) - rp.Sy * Bkz;
    const float Cx = sel(C, rp.kx) - rp.Sx * Ckz, Cy = sel(C, rp.ky) - rp.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    // the double-precision edge test is rare (an edge function exactly 0):
    // a wave-uniform branch keeps it off the common path
    const bool edge0 = U == 0.0f || V == 0.0f || W == 0.0f;
    if (__ballot(edge0) != 0ull && edge0) {
        double CxBy = (double)Cx * (double)By, CyBx = (double)Cy * (double)Bx;
        U = (float)(CxBy - CyBx);
        double AxCy = (double)Ax * (double)Cy, AyCx = (double)Ay * (double)Cx;
        V = (float)(AxCy - AyCx);
        double BxAy = (double)Bx * (double)Ay, ByAx = (double)By * (double)Ax;
        W = (float)(BxAy - ByAx);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    const float det = U + V + W;
    if (det == 0.0f) return false;
    const float Az = rp.Sz * Akz, Bz = rp.Sz * Bkz, Cz = rp.Sz * Ckz;
    const float T = U * Az + V * Bz + W * Cz;
    const float rcp = 1.0f / det;
    const float t = T * rcp;
    if (!(t >= tmin && t <= tmax)) return false;
    t_out = t;
    u_out = V * rcp;
    v_out = W * rcp;
    return true;
}

struct HitRec {
    float t, u, v;
    uint32_t gid, prim, inst;  // gid = 0xFFFFFFFF on a miss
};

// Relative bound (2^-21) on the rounding of a child slab distance q * a + b:
// a = 2^e * inv and b = (p - o) * inv each carry one rounding, inv one more
// and the fused multiply-add one, i.e. |error| < 4 eps (65535 |a| + |b|)
// (planes are at most 65504).
constexpr float kSlabErr = 4.76837158e-7f;  // 2^-21

// The ray's bounds over every node of the tree: the root's box [lo, hi]
// (sv.root_*) holds every node and every vertex, so along an axis no plane
// origin lies farther than M = max(|lo - o|, |hi - o|) from the ray's and no
// plane farther than X = hi - lo from its origin (and 2^-10 of that, rounded
// outward to fp16; the bound above has twice the room its four roundings need).
// Per ray instead of per node this saves 17 of the node step's instructions
// and visits no more nodes: against bounds of each node, shadow rays between
// points of the Cornell box 2.49 and 2.55 triangle tests, bounce rays of the
// 20,000-triangle caustics scene 0.21 and 0.21, of a 60,000-triangle terrain
// 6.33 and 6.32 (3.02, 1.48 and 6.37 with M + 2^17 2^e of the root for M).
//   err    2^-21 |1/d| (M + X) per axis: [t_near - err, t_far + err] contains
//          a child's true slab interval;
//   margin 2^-16 |1/d| M of the dominant axis.  A triangle's watertight t is
//          the mean of its vertices' t, weighted with the computed edge
//          functions.  Each term carries six roundings, the sums, the
//          reciprocal and the product four more: with z the farthest of the
//          vertices' t, at most |1/d| M, it is within 10 2^-24 z of the exact
//          mean, which lies in the box's interval of that axis.  The other
//          25-fold is for the weights' own roundings, which grow as a triangle
//          is seen edge-on.  Children are kept if they reach
//          [tmin - margin, tcur + margin], so a triangle whose computed t
//          undercuts the current best by that error is still tested.
LT_DEV void ray_bounds(const SceneView& sv, f3 o, RayPre& rp) {
    const f3 M = {fmaxf(fabsf(sv.root_lo[0] - o.x), fabsf(sv.root_hi[0] - o.x)),
                  fmaxf(fabsf(sv.root_lo[1] - o.y), fabsf(sv.root_hi[1] - o.y)),
                  fmaxf(fabsf(sv.root_lo[2] - o.z), fabsf(sv.root_hi[2] - o.z))};
    const f3 k = kSlabErr * mk3(fabsf(rp.inv.x), fabsf(rp.inv.y), fabsf(rp.inv.z));
    rp.err = {k.x * (M.x + sv.root_x[0]), k.y * (M.y + sv.root_x[1]), k.z * (M.z + sv.root_x[2])};
    rp.margin = sel({k.x * M.x, k.y * M.y, k.z * M.z}, rp.kz) * 32.0f;  // 2^-16 = 32 kSlabErr
}

// LDS-qualified so that stack accesses compile to ds_read / ds_write rather
// than flat accesses through the generic address space
typedef __attribute__((address_space(3))) uint32_t lds_u32;

struct TraceStack {
    lds_u32* lds;     // this thread's column: entry i at lds[i * kTraceBlock]
    lds_u32* q;       // its leaf queue, after the kLdsStack stack entries
    uint32_t* spill;  // this thread's spill area
    LT_DEV TraceStack(uint32_t* lds_col, uint32_t* spill_area)
        : lds((lds_u32*)lds_col), q((lds_u32*)lds_col + ltb::kLdsStack * kTraceBlock), spill(spill_area) {}
};

// entry i of the stack; a tree of at most kLdsStack + 1 levels (sv.deep_stack
// == 0, uniform) never leaves the LDS part
LT_DEV void stk_set(const SceneView& sv, const TraceStack& s, uint32_t i, uint32_t v) {
    if (sv.deep_stack && i >= (uint32_t)ltb::kLdsStack)
        s.spill[i - ltb::kLdsStack] = v;
    else
        s.lds[i * kTraceBlock] = v;
}
LT_DEV uint32_t stk_get(const SceneView& sv, const TraceStack& s, uint32_t i) {
    if (sv.deep_stack && i >= (uint32_t)ltb::kLdsStack) return s.spill[i - ltb::kLdsStack];
    return s.lds[i * kTraceBlock];
}

// a lane takes its next node while at most this many words of leaf groups are
// queued (0: only once every triangle it has hit the box of is tested)
#ifndef LT_NODE_PEND_MAX
#define LT_NODE_PEND_MAX (ltb::kLeafQueue - 8)
#endif
// a node step queues one group (2 words) more: the queue must hold it
static_assert(LT_NODE_PEND_MAX >= 0 && LT_NODE_PEND_MAX + 8 <= (int)ltb::kLeafQueue,
              "LT_NODE_PEND_MAX + 8 words exceed the per-lane LDS leaf queue");

// A node's internal children lie along its longest axis in slot order (the
// builder sorts them by their centres; the axis is the one of the largest
// exponent, the first of equals), so a ray that runs up the axis visits the
// hit ones from the lowest slot up and one that runs down it from the highest
// slot down: nearly front to back, without comparing their entry distances.
//
// A stack entry is the group of a node's hit internal children that still wait
// after the first: seven slots at most, because the first is the lowest
// (upward) or the highest (downward) hit one.
//   upward:   (child_base << 8) | slots (bits 1..7) | 1; lowest bit next
//   downward: (child_base - 1) << 8 | slots << 1 (bits 1..7); highest bit next
// Either way bit b is node (entry >> 8) + b, and the builder caps a BVH at
// 2^24 nodes.  One entry per tree level instead of one per child.
constexpr uint32_t kNoNode = 0xFFFFFFFFu;

// The traversal of one query as a state machine, so that a lane can take a
// new query as soon as its current one finishes (trace_step returns true).
struct TraceState {
    f3 o, d;
    RayPre rp;
    float tmin, tmax;
    float lo, hi;  // cull limits: tmin - margin, current best t + margin
    HitRec best;
    uint32_t sp;
    uint32_t next;           // node to visit next, or kNoNode
    uint32_t tri_base, tris; // leaf group being tested: bit i is triangle tri_base + i
    uint32_t qn;             // words of further leaf groups queued in LDS
};

LT_DEV void trace_init(const SceneView& sv, TraceState& s, f3 o, f3 d, float tmin, float tmax) {
    s.o = o;
    s.d = d;
    s.tmin = tmin;
    s.tmax = tmax;
    s.best.gid = 0xFFFFFFFFu;
    s.best.t = tmax;
    s.best.prim = s.best.inst = 0xFFFFFFFFu;
    s.best.u = s.best.v = 0.0f;
    s.rp = prep_ray(d);
    ray_bounds(sv, o, s.rp);
    s.lo = tmin - s.rp.margin;
    s.hi = tmax + s.rp.margin;
    s.sp = 0;
    s.qn = 0;
    s.tri_base = s.tris = 0u;
    // a NaN in the origin or the direction: no triangle can be hit, so no node
    // is visited.  The node step could not tell: to its sign test a NaN distance
    // is a hit, of every child of every node.  (A NaN in tmin or tmax drops that
    // limit; leaving such rays, and empty intervals, out here too, lo <= hi,
    // changes how the adjoint's replay is allocated registers: 78.9 -> 81.7 ms.)
    const float e = s.rp.err.x + s.rp.err.y + s.rp.err.z;
    s.next = sv.num_nodes != 0 && e == e ? 0u : kNoNode;
}

// Processes one BVH8 node (its children's boxes; the hit leaves' triangles are
// queued, the hit internal children pushed) and tests one queued triangle.
// any: finishes at the first hit in [tmin, tmax] (a per-lane flag; constant
// where trace_step's template argument gives it).  Counters are only updated
// when COUNT.
template <bool COUNT>
LT_DEV bool trace_step_dyn(const SceneView& sv, TraceState& s, const TraceStack& stk, bool any, uint32_t& n_nodes,
                           uint32_t& n_tris) {
    const f3 o = s.o;
    const RayPre& rp = s.rp;
    HitRec& best = s.best;
    if (s.next != kNoNode && (LT_NODE_PEND_MAX == 0 ? s.tris == 0u : s.qn <= (uint32_t)LT_NODE_PEND_MAX)) {
        if (COUNT) n_nodes++;
        // 32-bit byte offsets from the node array (scalar base + vector offset
        // addressing; the builder caps a BVH at 2^24 nodes)
        const char* nbase = (const char*)sv.nodes;
        const uint32_t noff = s.next * 128u;
        const float4 w0 = *(const float4*)(nbase + noff);
        const uint4 w1 = *(const uint4*)(nbase + (noff + 16u));
        // near / far planes by the ray octant: the plane vectors sit at
        // 16-byte slots 2..4 (qlo x, y, z) and 5..7 (qhi), so the octant picks
        // the load address instead of selecting between loaded words
        const bool negx = rp.inv.x < 0.0f, negy = rp.inv.y < 0.0f, negz = rp.inv.z < 0.0f;
        const uint32_t noff2 = noff + 48u;
        const uint4 qnx = *(const uint4*)(nbase + ((negx ? noff2 : noff) + 32u));
        const uint4 qfx = *(const uint4*)(nbase + ((negx ? noff : noff2) + 32u));
        const uint4 qny = *(const uint4*)(nbase + ((negy ? noff2 : noff) + 48u));
        const uint4 qfy = *(const uint4*)(nbase + ((negy ? noff : noff2) + 48u));
        const uint4 qnz = *(const uint4*)(nbase + ((negz ? noff2 : noff) + 64u));
        const uint4 qfz = *(const uint4*)(nbase + ((negz ? noff : noff2) + 64u));
        const uint32_t ew = __float_as_uint(w0.w);  // e.x, e.y, e.z, imask
        const int ex = (int)(int8_t)(ew & 0xFF), ey = (int)(int8_t)((ew >> 8) & 0xFF),
                  ez = (int)(int8_t)((ew >> 16) & 0xFF);
        const uint32_t imask = ew >> 24;
        const uint32_t child_base = w1.x, tri_base = w1.y;
        const uint32_t meta_lo = w1.z, meta_hi = w1.w;
        // Slab distances of the children: t = q * a + b per axis with
        // a = 2^e / d (exact, one ldexp) and b = (p - o) / d, widened by err
        const float ax = ldexpf(rp.inv.x, ex);
        const float ay = ldexpf(rp.inv.y, ey);
        const float az = ldexpf(rp.inv.z, ez);
        const float dx = w0.x - o.x, dy = w0.y - o.y, dz = w0.z - o.z;
        const float bnx = fmaf(dx, rp.inv.x, -rp.err.x), bfx = fmaf(dx, rp.inv.x, rp.err.x);
        const float bny = fmaf(dy, rp.inv.y, -rp.err.y), bfy = fmaf(dy, rp.inv.y, rp.err.y);
        const float bnz = fmaf(dz, rp.inv.z, -rp.err.z), bfz = fmaf(dz, rp.inv.z, rp.err.z);
        uint32_t miss = 0;  // the sign of t1 - t0 shifts in, child 7 first
#pragma unroll
        for (int c = 7; c >= 0; c--) {
            const int sh = (c & 1) * 16;
            const int wd = c >> 1;
            auto lane16 = [&](const uint4& q) {  // the fp16 plane; the fma below takes it as is
                const uint32_t w = wd == 0 ? q.x : (wd == 1 ? q.y : (wd == 2 ? q.z : q.w));
                return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> sh));
            };
            float t0 = fmaxf(fmaxf(fmaf(lane16(qnx), ax, bnx), fmaf(lane16(qny), ay, bny)), fmaf(lane16(qnz), az, bnz));
            float t1 = fminf(fminf(fmaf(lane16(qfx), ax, bfx), fmaf(lane16(qfy), ay, bfy)), fmaf(lane16(qfz), az, bfz));
            t0 = fmaxf(t0, s.lo);
            t1 = fminf(t1, s.hi);
            // (miss << 1) | sign(t1 - t0); equal distances give +0, a NaN (both
            // infinite; trace_init keeps others out) the default positive one: a hit
            miss = __builtin_amdgcn_alignbit(miss, __float_as_uint(t1 - t0), 31);
        }
        const uint32_t hit_int = imask & ~miss;
        // hit slots that are not internal: leaves, and (rarely, within the
        // rounding margin) empty slots, whose count of 0 queues nothing
        uint32_t hit_leaf = ~miss & ~imask & 0xFFu;
        if (hit_leaf) {
            uint32_t m = 0u;
            do {
                const int c = __builtin_ctz(hit_leaf);
                hit_leaf &= hit_leaf - 1;
                const uint32_t meta = ((c < 4 ? meta_lo : meta_hi) >> ((c & 3) * 8)) & 0xFF;
                m |= ((1u << (meta & 7u)) - 1u) << (meta >> 3);  // offsets and counts: at most 32 triangles
            } while (hit_leaf);
            if (s.tris == 0u) {
                s.tri_base = tri_base;
                s.tris = m;
            } else if (m) {
                stk.q[s.qn * kTraceBlock] = tri_base;
                stk.q[(s.qn + 1u) * kTraceBlock] = m;
                s.qn += 2u;
            }
        }
        // the longest axis' direction decides the order of the children
        const bool up = ez > max(ex, ey) ? !negz : (ey > ex ? !negy : !negx);
        if (hit_int) {
            const uint32_t first = up ? (uint32_t)__builtin_ctz(hit_int) : 31u - (uint32_t)__builtin_clz(hit_int);
            const uint32_t rest = hit_int ^ (1u << first);
            s.next = child_base + first;
            if (rest) {
                stk_set(sv, stk, s.sp, up ? ((child_base << 8) | rest | 1u) : (((child_base - 1u) << 8) | (rest << 1)));
                s.sp++;
            }
        } else if (s.sp != 0u) {
            const uint32_t e = stk_get(sv, stk, s.sp - 1u);
            const uint32_t slots = e & 0xFEu;
            const uint32_t r =
                (e & 1u) ? (uint32_t)__builtin_ctz(slots) : 31u - (uint32_t)__builtin_clz(slots);
            const uint32_t left = e ^ (1u << r);
            if (left & 0xFEu)
                stk_set(sv, stk, s.sp - 1u, left);
            else
                s.sp--;
            s.next = (e >> 8) + r;
        } else {
            s.next = kNoNode;
        }
    }
    // One queued triangle per lane and step: a node step and a triangle test
    // share the step instead of the wave looping over the most leaf hits of
    // any lane.  The other queued triangles wait for the next steps, which
    // only delays the shrinking of the cull limit (culling stays
    // conservative); an any-hit query ends at its first hit.
    if (s.tris != 0u) {
        const uint32_t b = (uint32_t)__builtin_ctz(s.tris);
        s.tris &= s.tris - 1u;
        const float4* tp = (const float4*)(sv.tris + (size_t)(s.tri_base + b));
        const float4 a = tp[0], bb = tp[1], cc = tp[2];
        if (COUNT) n_tris++;
        if (s.tris == 0u && s.qn != 0u) {
            s.qn -= 2u;
            s.tri_base = stk.q[s.qn * kTraceBlock];
            s.tris = stk.q[(s.qn + 1u) * kTraceBlock];
        }
        float t, u, v;
        if (isect_tri(mk3(a.x, a.y, a.z), mk3(a.w, bb.x, bb.y), mk3(bb.z, bb.w, cc.x), o, rp, s.tmin, s.tmax, t, u, v)) {
            const uint32_t gid = __float_as_uint(cc.y);
            if (any || t < best.t || (t == best.t && gid < best.gid)) {
                best.t = t;
                best.u = u;
                best.v = v;
                best.gid = gid;
                best.prim = __float_as_uint(cc.z);
                best.inst = __float_as_uint(cc.w);
                s.hi = t + rp.margin;
                if (any) return true;
            }
        }
    }
    return s.next == kNoNode && s.tris == 0u;
}

template <bool ANY, bool COUNT>
LT_DEV bool trace_step(const SceneView& sv, TraceState& s, const TraceStack& stk, uint32_t& n_nodes,
                       uint32_t& n_tris) {
    return trace_step_dyn<COUNT>(sv, s, stk, ANY, n_nodes, n_tris);
}

// Streams the queries [0, n_items) of a queue through one wave: every lane
// steps its own query one node at a time, and once sv.refill_min lanes are
// idle they hand out their results together and take new queries of the wave's
// tiles (dev_work.h), so the wave stays full however uneven the traversal
// lengths are and nothing but the step runs between two refills.
// load(item, o, d, tmin, tmax, any) returns a tag handed to finish(tag, state);
// any says whether the query is an any-hit one (ANY_MASK 1: none is, 2: every
// one is, 3: one by one).
template <int ANY_MASK, bool COUNT, class Load, class Finish>
LT_DEV void trace_stream(const SceneView& sv, const TraceStack& stk, uint32_t n_items, uint32_t* work, Load load,
                         Finish finish, uint32_t& n_nodes, uint32_t& n_tris) {
    TraceState s;
    uint32_t tag = 0;
    bool has = false, out = false, any = ANY_MASK == 2;
    WaveTiles wt = wave_tiles(n_items, work);
    for (;;) {
        const unsigned long long idle = __ballot(!has);
        const uint32_t n_idle = (uint32_t)__popcll(idle);
        if (n_idle == 64u || (!wt.done && n_idle >= sv.refill_min)) {
            if (out) finish(tag, s);
            out = out && has;
            if (n_idle == 64u && wt.done) break;
            uint32_t item = 0u;
            if (take_items(wt, idle, item)) {
                f3 o, d;
                float tmin, tmax;
                bool a = ANY_MASK == 2;
                tag = load(item, o, d, tmin, tmax, a);
                if (ANY_MASK == 3) any = a;
                trace_init(sv, s, o, d, tmin, tmax);
                has = true;
            }
            if (__ballot(has) == 0ull) break;
        }
        if (has && trace_step_dyn<COUNT>(sv, s, stk, ANY_MASK == 1 ? false : (ANY_MASK == 2 ? true : any), n_nodes, n_tris)) {
            has = false;
            out = true;
        }
    }
}

// Paths streamed through a wave: a lane owns a path, and lanes whose ray has
// ended wait until kPathWait of them do (or half of the lanes still under way),
// so the wave keeps stepping the other rays; then the waiting lanes shade
// together and those whose path ended take the next item.  Only for paths whose
// shading is short: shading in smaller groups costs more of it, and its memory
// latencies stop the whole wave more often.  SPPM's light pass (13 of 64 lanes
// active when a wave shaded after the longest of its 64 rays): 14.85 ms per 8
// frames before, 16.1 / 14.6 / 14.1 / 13.9 / 13.9 ms when 8 / 16 / 24 / 32 / 48
// lanes wait; the BDPT walk, which stores 16 words per vertex, 19.9 ms before
// and 22.5 ms with 32, so it is not used there.
//   shade(t, r)      the lane's ray has ended (t.best): folds it in and sets
//                    the next ray r; false if the path has ended
//   begin(item, r)   starts the path of an item; false if the item has none
#ifndef LT_PATH_WAIT
#define LT_PATH_WAIT 32
#endif
constexpr uint32_t kPathWait = LT_PATH_WAIT;

struct PathRay {
    f3 o, d;
    float tmin, tmax;
};

template <bool COUNT, class Shade, class Begin>
LT_DEV void stream_paths(const SceneView& sv, const TraceStack& stk, WaveTiles wt, Shade shade, Begin begin, Ctr& c) {
    TraceState t;
    bool has = false, out = false, path = false;
    for (;;) {
        const unsigned long long run = __ballot(has);
        const uint32_t n_run = (uint32_t)__popcll(run);
        const uint32_t n_wait = (uint32_t)__popcll(wt.done ? __ballot(out) : ~run);
        if (n_wait >= kPathWait || n_wait >= n_run) {
            PathRay r;
            bool next = false;
            if (out) {
                next = shade(t, r);
                path = next;
                out = false;
            }
            uint32_t item = 0u;
            if (take_items(wt, __ballot(!path), item)) {
                next = begin(item, r);
                path = next;
            }
            if (next) {
                trace_init(sv, t, r.o, r.d, r.tmin, r.tmax);
                has = true;
            }
            if (__ballot(has) == 0ull) {
                if (wt.done) break;
                continue;
            }
        }
        if (has) {
            if (trace_step<false, COUNT>(sv, t, stk, c.nodes, c.tris)) {
                has = false;
                out = true;
            }
        }
    }
}

// Whole query on one lane.
template <bool ANY, bool COUNT>
LT_DEV bool trace_bvh(const SceneView& sv, f3 o, f3 d, float tmin, float tmax, HitRec& best, const TraceStack& stk,
                      uint32_t& n_nodes, uint32_t& n_tris) {
    TraceState s;
    trace_init(sv, s, o, d, tmin, tmax);
    while (!trace_step<ANY, COUNT>(sv, s, stk, n_nodes, n_tris)) {
    }
    best = s.best;
    return s.best.gid != 0xFFFFFFFFu;
}

}  // namespace ltd
