// bvh_build.hip — GPU BVH build: a binary tree collapsed to a quantised BVH8 (gfx950).
//
// Replaces the driver build behind Integrator::create_accel ->
// vk::build_blas / vk::build_tlas (src/RayTracer/Integrator.cpp:137-160,
// src/Framework/AccelerationStructure.cpp:171-315).  Stages:
//   1. k_make_tris     : 48-B triangle records + centroid bounds (atomics)
//   2. k_morton        : 30-bit Morton codes of the centroids
//   3. radix sort      : (morton, triangle) pairs, rocPRIM radix sort (bits 0..29)
//   4. binary tree     : PLOC (default): rounds of k_ploc_merge and
//                        k_ploc_compact, the last ones in k_ploc_tail; boxes,
//                        counts and the SAH tables of a node are made with it.
//                        LBVH: k_karras (Karras 2012, one thread per node),
//                        then k_refit bottom-up with arrival counters
//      SAH tables      : dynamic programme over the binary tree (Ylitie,
//                        Karras & Laine 2017): per node the cheapest cover of
//                        its subtree by at most i = 1..8 BVH8 subtree roots
//   5. k_collapse      : top-down BVH8 collapse, one thread per BVH8 node and
//                        level; a node's children are the roots the programme
//                        chose (or, greedy, the expansion of the child with the
//                        largest surface area), subtrees of <= max_leaf
//                        triangles become leaves; fp16 planes, 128-B nodes
//   6. k_check         : every child and leaf range in bounds
// What bounds it is not work but steps: launches, looks of the host at device
// counts, fences and atomics on shared lines.  250k triangles: 12.2 ms with a
// launch and a host look per round and level, a pass each for counts, ranges
// and tables and a host check of the nodes; 1.7 ms now (1M: 29.9 and 2.5 ms).
// These are repeated builds: a context's first one also allocates the
// workspace (1M: 6.5 ms).
#include <hip/hip_runtime.h>

#include <rocprim/device/device_radix_sort.hpp>
#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>

#include "context.h"

using ltb::Node8;
using ltb::TriRec;

namespace {

struct Box {
    float lo[3], hi[3];
};
constexpr uint32_t kLine = 32;  // words of a cache line

__device__ __forceinline__ uint32_t f2ord(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// object-to-world point of the transform rows xf (3 x 4), evaluated without
// contraction in the order the host replay uses
__device__ __forceinline__ void xf_point(const float* __restrict__ xf, const float* p, float* o) {
#pragma clang fp contract(off)
    for (int i = 0; i < 3; i++) o[i] = ((xf[4 * i] * p[0] + xf[4 * i + 1] * p[1]) + xf[4 * i + 2] * p[2]) + xf[4 * i + 3];
}

// One thread per triangle g of the flattened triangle list (mesh by mesh,
// instances of one geometry each with their own triangles): the mesh by
// binary search over the meshes' first triangles; vertices in world space
// through the mesh's transform, the flattening that gives one BVH the
// instance semantics of the reference's TLAS (Integrator.cpp:147-158).
__global__ void k_make_tris(const lt_vertex* __restrict__ vtx, const uint32_t* __restrict__ idx,
                            const lt_prim_mesh_info* __restrict__ prims, const uint32_t* __restrict__ tri_start,
                            const float* __restrict__ xf, uint32_t nprims, uint32_t ntri, TriRec* __restrict__ out,
                            uint32_t* __restrict__ cbounds /* 6 ordered uints, kLine words apart */) {
    float clo[3] = {INFINITY, INFINITY, INFINITY}, chi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < ntri; g += gridDim.x * blockDim.x) {
        uint32_t lo = 0, hi = nprims;  // last mesh whose first triangle is <= g
        while (hi - lo > 1) {
            uint32_t mid = (lo + hi) >> 1;
            if (tri_start[mid] <= g)
                lo = mid;
            else
                hi = mid;
        }
        const lt_prim_mesh_info pi = prims[lo];
        const uint32_t prim = g - tri_start[lo];
        const uint32_t io = pi.index_offset + 3 * prim;
        TriRec r;
        const float* a = vtx[idx[io] + pi.vertex_offset].pos;
        const float* b = vtx[idx[io + 1] + pi.vertex_offset].pos;
        const float* c = vtx[idx[io + 2] + pi.vertex_offset].pos;
        if (xf) {
            const float* m = xf + (size_t)kXfFloats * lo;
            xf_point(m, a, r.v0);
            xf_point(m, b, r.v1);
            xf_point(m, c, r.v2);
        } else {
            for (int k = 0; k < 3; k++) {
                r.v0[k] = a[k];
                r.v1[k] = b[k];
                r.v2[k] = c[k];
            }
        }
        for (int k = 0; k < 3; k++) {
            const float cen = (r.v0[k] + r.v1[k] + r.v2[k]) * (1.0f / 3.0f);
            clo[k] = fminf(clo[k], cen);
            chi[k] = fmaxf(chi[k], cen);
        }
        r.gid = g;
        r.prim = prim;
        r.inst = lo;
        out[g] = r;
    }
    // workgroup reduction of the centroid bounds, then one atomic per workgroup
    // and value, each value on a cache line of its own (an atomic per wave on
    // one line, 8-11 ns each, was most of 0.30 ms for 250k triangles)
    __shared__ float red[16][6];
    for (int k = 0; k < 3; k++) {
        float l = clo[k], h = chi[k];
        for (int o = 32; o > 0; o >>= 1) {
            l = fminf(l, __shfl_xor(l, o));
            h = fmaxf(h, __shfl_xor(h, o));
        }
        if ((threadIdx.x & 63) == 0) {
            red[threadIdx.x >> 6][k] = l;
            red[threadIdx.x >> 6][3 + k] = h;
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        float v = red[0][threadIdx.x];
        for (uint32_t w = 1; w < blockDim.x / 64u; w++)
            v = threadIdx.x < 3 ? fminf(v, red[w][threadIdx.x]) : fmaxf(v, red[w][threadIdx.x]);
        if (threadIdx.x < 3)
            atomicMin(&cbounds[threadIdx.x * kLine], f2ord(v));
        else
            atomicMax(&cbounds[threadIdx.x * kLine], f2ord(v));
    }
}

// fp16 bit patterns of non-negative plane values, rounded outward (the
// largest fp16 <= x / the smallest fp16 >= x, both within [0, 65504]): the
// double -> float -> fp16 conversion lands on one of the two fp16 values
// around x, and one step along the (monotone) bit pattern fixes the side.
__device__ __forceinline__ float f16_value(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
__device__ __forceinline__ uint16_t f16_floor(double x) {
    if (!(x > 0.0)) return 0;
    if (x >= 65504.0) return 0x7BFF;
    uint16_t h = __builtin_bit_cast(uint16_t, (_Float16)(float)x);
    if ((double)f16_value(h) > x) h -= 1;
    return h;
}
__device__ __forceinline__ uint16_t f16_ceil(double x) {
    if (!(x > 0.0)) return 0;
    if (x >= 65504.0) return 0x7BFF;
    uint16_t h = __builtin_bit_cast(uint16_t, (_Float16)(float)x);
    if ((double)f16_value(h) < x) h += 1;
    return h;
}

__device__ __forceinline__ uint32_t expand_bits(uint32_t v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

__global__ void k_morton(const TriRec* __restrict__ tris, uint32_t n, const uint32_t* __restrict__ cb,
                         uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
    uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    const TriRec r = tris[g];
    uint32_t code = 0;
    uint32_t q[3];
    for (int k = 0; k < 3; k++) {
        float lo = ord2f(cb[k * kLine]), hi = ord2f(cb[(3 + k) * kLine]);
        float cen = (r.v0[k] + r.v1[k] + r.v2[k]) * (1.0f / 3.0f);
        float ext = hi - lo;
        float t = ext > 0.0f ? (cen - lo) / ext : 0.5f;
        q[k] = (uint32_t)fminf(fmaxf(t * 1024.0f, 0.0f), 1023.0f);
    }
    code = (expand_bits(q[0]) << 2) | (expand_bits(q[1]) << 1) | expand_bits(q[2]);
    keys[g] = code;
    vals[g] = g;
}

__device__ __forceinline__ int delta(const uint32_t* __restrict__ k, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    uint32_t a = k[i], b = k[j];
    if (a == b) return 32 + __clz((uint32_t)(i ^ j));
    return __clz(a ^ b);
}

// Karras 2012, "Maximizing parallelism in the construction of BVHs, octrees
// and k-d trees".  Children: bit 31 set = leaf (index into sorted order).
__global__ void k_karras(const uint32_t* __restrict__ keys, int n, uint32_t* __restrict__ left,
                         uint32_t* __restrict__ right, uint32_t* __restrict__ parent_int,
                         uint32_t* __restrict__ parent_leaf, uint32_t* __restrict__ range_lo,
                         uint32_t* __restrict__ range_hi) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = delta(keys, n, i, i - d);
    int lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = delta(keys, n, i, j);
    int s = 0;
    int t = l;
    do {
        t = (t + 1) >> 1;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    int gamma = i + s * d + (d < 0 ? -1 : 0);
    int lo = min(i, j), hi = max(i, j);
    uint32_t lc = (lo == gamma) ? (0x80000000u | (uint32_t)gamma) : (uint32_t)gamma;
    uint32_t rc = (hi == gamma + 1) ? (0x80000000u | (uint32_t)(gamma + 1)) : (uint32_t)(gamma + 1);
    left[i] = lc;
    right[i] = rc;
    range_lo[i] = (uint32_t)lo;
    range_hi[i] = (uint32_t)hi;
    if (lc & 0x80000000u)
        parent_leaf[lc & 0x7fffffffu] = (uint32_t)i;
    else
        parent_int[lc] = (uint32_t)i;
    if (rc & 0x80000000u)
        parent_leaf[rc & 0x7fffffffu] = (uint32_t)i;
    else
        parent_int[rc] = (uint32_t)i;
}

__device__ __forceinline__ Box tri_box(const TriRec& r) {
    Box b;
    for (int k = 0; k < 3; k++) {
        b.lo[k] = fminf(r.v0[k], fminf(r.v1[k], r.v2[k]));
        b.hi[k] = fmaxf(r.v0[k], fmaxf(r.v1[k], r.v2[k]));
    }
    return b;
}

__device__ __forceinline__ float half_area(const Box& b) {
    float dx = b.hi[0] - b.lo[0], dy = b.hi[1] - b.lo[1], dz = b.hi[2] - b.lo[2];
    return dx * dy + dy * dz + dz * dx;
}

// ---- PLOC binary tree (Meister and Bittner 2018, "Parallel locally-ordered
// clustering for bounding volume hierarchy construction") ----
// The clusters start as the Morton-sorted triangles.  Each round, every
// cluster finds the neighbour within kPlocRadius positions whose union box has
// the smallest surface area; mutual nearest neighbours merge into a new
// internal node (allocated from n - 2 down, so the last merge is the root 0
// and a parent's index is below its children's), and the survivors are
// compacted in order.  Ties are broken by the pair's indices, a strict order
// under which the globally closest pair is mutual, so every round merges.
#ifndef LT_PLOC_RADIUS
#define LT_PLOC_RADIUS 16
#endif
constexpr int kPlocRadius = LT_PLOC_RADIUS;

__device__ __forceinline__ Box box_union(const Box& a, const Box& b) {
    Box r;
    for (int k = 0; k < 3; k++) {
        r.lo[k] = fminf(a.lo[k], b.lo[k]);
        r.hi[k] = fmaxf(a.hi[k], b.hi[k]);
    }
    return r;
}

// Both builders' trees: bit 31 of a child marks a leaf (index into the Morton
// order).  The tables of the SAH programme (below) and the triangle counts of
// a merged node are made where it is made: its children are complete, so no
// pass over the finished tree is needed (a bottom-up pass with a fence and
// an atomic per node took 1.5 ms for the counts and 2.1 ms for the boxes and
// tables of 250k triangles: fences of device scope cross the 8 XCDs' L2s).
// SAH weights of a BVH8 node visit and of a triangle test (a watertight
// test costs about half a node step)
#ifndef LT_SAH_TRI_COST
#define LT_SAH_TRI_COST 0.5f
#endif
constexpr float kSahNode = 1.0f;
constexpr float kSahTri = LT_SAH_TRI_COST;
constexpr uint8_t kDecLeaf = 0xFF;

// The dynamic programme at internal node p (children a, b):
//   R(p, i) = cheapest cover of p's subtree by at most i subtree roots,
//   R(p, 1) = min(leaf cost (<= max_leaf triangles), A(p) kSahNode + min_k R(a, k) + R(b, 8 - k)),
//   R(p, i) = min(R(p, i - 1), min_k R(a, k) + R(b, i - k)),  i = 2..8,
// a binary leaf costing A kSahTri for any i.  dec[p][0] = kDecLeaf or the k of
// the node's own 8 roots; dec[p][i - 1] = 0 (fewer roots) or the k of the split.
__device__ void sah_node(const float* ra, const float* rb, const Box& pb, uint32_t cnt, uint32_t max_leaf,
                         float* __restrict__ out, uint8_t* __restrict__ d) {
    float node = INFINITY;
    uint8_t node_k = 1;
#pragma unroll
    for (int k = 1; k < 8; k++) {
        const float v = ra[k - 1] + rb[8 - k - 1];
        if (v < node) {
            node = v;
            node_k = (uint8_t)k;
        }
    }
    node += half_area(pb) * kSahNode;
    const float leaf = cnt <= max_leaf ? half_area(pb) * kSahTri * (float)cnt : INFINITY;
    out[0] = leaf <= node ? leaf : node;
    d[0] = leaf <= node ? kDecLeaf : node_k;
#pragma unroll
    for (int i = 2; i <= 8; i++) {
        float best = out[i - 2];
        uint8_t bk = 0;
#pragma unroll
        for (int k = 1; k < i; k++) {
            const float v = ra[k - 1] + rb[i - k - 1];
            if (v < best) {
                best = v;
                bk = (uint8_t)k;
            }
        }
        out[i - 1] = best;
        d[i - 1] = bk;
    }
}

// a node's table and decisions, written as whole words
__device__ __forceinline__ void sah_store(float* __restrict__ R, uint8_t* __restrict__ dec, uint32_t p,
                                          const float* out, const uint8_t* d) {
    float4* r = (float4*)(R + (size_t)p * 8);
    r[0] = make_float4(out[0], out[1], out[2], out[3]);
    r[1] = make_float4(out[4], out[5], out[6], out[7]);
    uint2 w;
    w.x = d[0] | (d[1] << 8) | (d[2] << 16) | ((uint32_t)d[3] << 24);
    w.y = d[4] | (d[5] << 8) | (d[6] << 16) | ((uint32_t)d[7] << 24);
    *(uint2*)(dec + (size_t)p * 8) = w;
}


struct PlocTree {
    uint32_t *left, *right, *cnt;
    Box *ibox, *lbox;
    float* R;      // NULL: no SAH tables
    uint8_t* dec;
    uint32_t n, max_leaf;
};

// internal node idx of the clusters a (box ba) and b
__device__ void ploc_node(const PlocTree& T, uint32_t idx, uint32_t a, const Box& ba, uint32_t b, const Box& bb,
                          const Box& u) {
    T.left[idx] = a;
    T.right[idx] = b;
    const uint32_t c = ((a & 0x80000000u) ? 1u : T.cnt[a]) + ((b & 0x80000000u) ? 1u : T.cnt[b]);
    T.cnt[idx] = c;
    T.ibox[idx] = u;
    if (!T.R) return;
    float ra[8], rb[8], out[8];
    uint8_t d[8];
    auto load = [&](uint32_t k, const Box& bx, float* t) {
        if (k & 0x80000000u) {
            const float v = half_area(bx) * kSahTri;
            for (int i = 0; i < 8; i++) t[i] = v;
        } else {
            const float4* r = (const float4*)(T.R + (size_t)k * 8);
            const float4 x = r[0], y = r[1];
            t[0] = x.x, t[1] = x.y, t[2] = x.z, t[3] = x.w;
            t[4] = y.x, t[5] = y.y, t[6] = y.z, t[7] = y.w;
        }
    };
    load(a, ba, ra);
    load(b, bb, rb);
    sah_node(ra, rb, u, c, T.max_leaf, out, d);
    sah_store(T.R, T.dec, idx, out, d);
}

__global__ void k_ploc_init(const TriRec* __restrict__ tris, const uint32_t* __restrict__ sorted, uint32_t n,
                            uint32_t* __restrict__ cl_node, Box* __restrict__ cl_box, Box* __restrict__ lbox) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const Box b = tri_box(tris[sorted[i]]);
    cl_node[i] = 0x80000000u | i;
    cl_box[i] = b;
    lbox[i] = b;
}

// A box in LDS: six planes, so that neighbouring lanes read neighbouring words.
template <int N>
struct LdsBoxes {
    float v[6][N];
    __device__ void put(int i, const Box& b) {
        for (int k = 0; k < 3; k++) {
            v[k][i] = b.lo[k];
            v[3 + k][i] = b.hi[k];
        }
    }
    __device__ Box get(int i) const {
        Box b;
        for (int k = 0; k < 3; k++) {
            b.lo[k] = v[k][i];
            b.hi[k] = v[3 + k][i];
        }
        return b;
    }
};

// The nearest neighbour of cluster i among [0, m) within the radius: (area,
// lower index, higher index) lexicographically smallest.  Indices are offset by
// `at` in the LDS array.
template <int N>
__device__ uint32_t ploc_nearest(const LdsBoxes<N>& bx, int i, int m, int at) {
    const Box bi = bx.get(i - at);
    const int lo = max(0, i - kPlocRadius), hi = min(m - 1, i + kPlocRadius);
    float best = INFINITY;
    uint32_t bj = (uint32_t)i, bmin = 0xFFFFFFFFu, bmax = 0xFFFFFFFFu;
    for (int j = lo; j <= hi; j++) {
        if (j == i) continue;
        const float a = half_area(box_union(bi, bx.get(j - at)));
        const uint32_t pmin = (uint32_t)min(i, j), pmax = (uint32_t)max(i, j);
        if (a < best || (a == best && (pmin < bmin || (pmin == bmin && pmax < bmax)))) {
            best = a;
            bj = (uint32_t)j;
            bmin = pmin;
            bmax = pmax;
        }
    }
    return bj;
}

// Rounds run on a cluster count that stays on the device (m[r] before round r);
// the host only bounds the grid.  Once m[r] is at most kPlocTail a round does
// nothing and k_ploc_tail finishes.
constexpr uint32_t kPlocBlock = 256;
constexpr uint32_t kPlocTail = 2048;
constexpr int kPlocHalo = 2 * kPlocRadius;  // a neighbour's own neighbours

// Nearest neighbours and merges of one round: mutual pairs merge at the lower
// index, the other cluster's node becomes kGone; survivors counted per block.
constexpr uint32_t kGone = 0xFFFFFFFFu;
__global__ __launch_bounds__(kPlocBlock) void k_ploc_merge(PlocTree T, const uint32_t* __restrict__ cl_node,
                                                           const Box* __restrict__ cl_box,
                                                           const uint32_t* __restrict__ m_of, uint32_t round,
                                                           uint32_t* __restrict__ ctr, uint32_t* __restrict__ out_node,
                                                           Box* __restrict__ out_box, uint32_t* __restrict__ kept) {
    constexpr int W = (int)kPlocBlock + 2 * kPlocHalo;
    __shared__ LdsBoxes<W> bx;
    __shared__ uint32_t nn[kPlocBlock + 2 * kPlocRadius];
    __shared__ uint32_t s_merge, s_keep, s_base;
    const int m = (int)m_of[round];
    const int base = (int)(blockIdx.x * kPlocBlock);
    if (m <= (int)kPlocTail || base >= m) return;
    const int at = base - kPlocHalo;
    for (int k = (int)threadIdx.x; k < W; k += (int)kPlocBlock)
        if (at + k >= 0 && at + k < m) bx.put(k, cl_box[at + k]);
    if (threadIdx.x == 0) s_merge = s_keep = 0u;
    __syncthreads();
    for (int k = (int)threadIdx.x; k < (int)kPlocBlock + 2 * kPlocRadius; k += (int)kPlocBlock) {
        const int i = base - kPlocRadius + k;
        if (i >= 0 && i < m) nn[k] = ploc_nearest(bx, i, m, at);
    }
    __syncthreads();
    const int i = base + (int)threadIdx.x;
    const bool in = i < m;
    const int j = in ? (int)nn[threadIdx.x + kPlocRadius] : 0;
    const bool mutual = in && j != i && (int)nn[j - base + kPlocRadius] == i;
    const bool merge = mutual && i < j, keep = in && !(mutual && i > j);
    // one atomic per block for the node indices, n - 2 downwards
    uint32_t rank = 0u;
    if (merge) rank = atomicAdd(&s_merge, 1u);
    if (keep) atomicAdd(&s_keep, 1u);
    __syncthreads();
    if (threadIdx.x == 0) {
        s_base = s_merge ? atomicAdd(ctr, s_merge) : 0u;
        kept[blockIdx.x] = s_keep;
    }
    __syncthreads();
    if (!in) return;
    const uint32_t a = cl_node[i];
    const Box ba = bx.get(i - at);
    if (merge) {
        const uint32_t idx = T.n - 2u - (s_base + rank), b = cl_node[j];
        const Box bb = bx.get(j - at), u = box_union(ba, bb);
        ploc_node(T, idx, a, ba, b, bb, u);
        out_node[i] = idx;
        out_box[i] = u;
    } else {
        out_node[i] = keep ? a : kGone;
        if (keep) out_box[i] = ba;
    }
}

// the survivors in order; m[round + 1]
__global__ __launch_bounds__(kPlocBlock) void k_ploc_compact(const uint32_t* __restrict__ in_node,
                                                             const Box* __restrict__ in_box, uint32_t* __restrict__ m_of,
                                                             uint32_t round, const uint32_t* __restrict__ kept,
                                                             uint32_t* __restrict__ out_node, Box* __restrict__ out_box) {
    __shared__ uint32_t s_sum[kPlocBlock / 64], s_cnt[kPlocBlock / 64];
    const uint32_t m = m_of[round];
    if (m <= kPlocTail) {
        if (blockIdx.x == 0 && threadIdx.x == 0) m_of[round + 1] = m;
        return;
    }
    const uint32_t blocks = (m + kPlocBlock - 1u) / kPlocBlock;
    if (blockIdx.x >= blocks) return;
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    uint32_t before = 0u;  // survivors of the blocks before this one
    for (uint32_t k = threadIdx.x; k < blockIdx.x; k += kPlocBlock) before += kept[k];
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o);
    const uint32_t i = blockIdx.x * kPlocBlock + threadIdx.x;
    const uint32_t node = i < m ? in_node[i] : kGone;
    const unsigned long long live = __ballot(node != kGone);
    if (lane == 0u) {
        s_sum[w] = before;
        s_cnt[w] = (uint32_t)__popcll(live);
    }
    __syncthreads();
    uint32_t pos = 0u, total = 0u;
    for (uint32_t k = 0; k < kPlocBlock / 64; k++) {
        total += s_sum[k] + s_cnt[k];
        pos += s_sum[k] + (k < w ? s_cnt[k] : 0u);
    }
    if (node != kGone) {
        pos += (uint32_t)__popcll(live & ((1ull << lane) - 1ull));
        out_node[pos] = node;
        out_box[pos] = in_box[i];
    }
    if (blockIdx.x == blocks - 1u && threadIdx.x == 0) m_of[round + 1] = total;
}

// The last rounds, at most kPlocTail clusters, in one workgroup's LDS (a launch
// per round and step cost about 50 us a round, and 30 of 53 rounds of 250k
// triangles are these).  ok = 0 if a round merged nothing.
constexpr uint32_t kTailBlock = 1024;
__global__ __launch_bounds__(kTailBlock) void k_ploc_tail(PlocTree T, const uint32_t* __restrict__ cl_node,
                                                          const Box* __restrict__ cl_box,
                                                          const uint32_t* __restrict__ m_of, uint32_t round,
                                                          uint32_t* __restrict__ ctr, uint32_t* __restrict__ ok) {
    constexpr int P = (int)(kPlocTail / kTailBlock);
    __shared__ LdsBoxes<(int)kPlocTail> bx;
    __shared__ uint32_t node[kPlocTail];
    __shared__ uint16_t nn[kPlocTail];
    __shared__ uint32_t s_keep[kTailBlock / 64], s_merge[kTailBlock / 64];
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    uint32_t m = m_of[round], done = *ctr;
    for (uint32_t i = threadIdx.x; i < m; i += kTailBlock) {
        node[i] = cl_node[i];
        bx.put((int)i, cl_box[i]);
    }
    __syncthreads();
    // a thread's clusters are neighbours, so that the survivors keep their order
    while (m > 1u) {
        for (uint32_t i = threadIdx.x; i < m; i += kTailBlock) nn[i] = (uint16_t)ploc_nearest(bx, (int)i, (int)m, 0);
        __syncthreads();
        uint32_t c_node[P], n_keep = 0u, n_merge = 0u;
        Box c_box[P];
        bool c_keep[P], c_merge[P];
        uint32_t c_j[P];
#pragma unroll
        for (int k = 0; k < P; k++) {
            const uint32_t i = threadIdx.x * P + k;
            const uint32_t j = i < m ? nn[i] : 0u;
            const bool mutual = i < m && j != i && nn[j] == i;
            c_merge[k] = mutual && i < j;
            c_keep[k] = i < m && !(mutual && i > j);
            c_j[k] = j;
            n_keep += c_keep[k] ? 1u : 0u;
            n_merge += c_merge[k] ? 1u : 0u;
        }
        uint32_t sk = n_keep, sm = n_merge;  // inclusive scans over the workgroup
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t a = __shfl_up(sk, (unsigned)o), b = __shfl_up(sm, (unsigned)o);
            if ((int)lane >= o) {
                sk += a;
                sm += b;
            }
        }
        if (lane == 63u) {
            s_keep[w] = sk;
            s_merge[w] = sm;
        }
        __syncthreads();
        uint32_t pk = sk - n_keep, pm = sm - n_merge, tk = 0u, tm = 0u;
        for (uint32_t k = 0; k < kTailBlock / 64; k++) {
            pk += k < w ? s_keep[k] : 0u;
            pm += k < w ? s_merge[k] : 0u;
            tk += s_keep[k];
            tm += s_merge[k];
        }
        if (tm == 0u) {  // uniform: no pair of this round is mutual
            if (threadIdx.x == 0) *ok = 0u;
            return;
        }
#pragma unroll
        for (int k = 0; k < P; k++) {
            const uint32_t i = threadIdx.x * P + k;
            if (!c_keep[k]) continue;
            c_node[k] = node[i];
            c_box[k] = bx.get((int)i);
            if (c_merge[k]) {
                const uint32_t idx = T.n - 2u - (done + pm++), b = node[c_j[k]];
                const Box bb = bx.get((int)c_j[k]), u = box_union(c_box[k], bb);
                ploc_node(T, idx, c_node[k], c_box[k], b, bb, u);
                c_node[k] = idx;
                c_box[k] = u;
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < P; k++)
            if (c_keep[k]) {
                node[pk] = c_node[k];
                bx.put((int)pk, c_box[k]);
                pk++;
            }
        m = tk;
        done += tm;
        __syncthreads();
    }
}

// bottom-up refit: second arrival at a node computes its box (and, when R is
// given, the SAH programme of the node)
__global__ void k_refit(const TriRec* __restrict__ tris, const uint32_t* __restrict__ sorted, int n,
                        const uint32_t* __restrict__ left, const uint32_t* __restrict__ right,
                        const uint32_t* __restrict__ parent_int, const uint32_t* __restrict__ parent_leaf,
                        uint32_t* __restrict__ flags, Box* __restrict__ ibox, Box* __restrict__ lbox,
                        const uint32_t* __restrict__ rlo, const uint32_t* __restrict__ rhi, uint32_t max_leaf,
                        float* __restrict__ R, uint8_t* __restrict__ dec, uint32_t* __restrict__ cnt) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    lbox[i] = tri_box(tris[sorted[i]]);
    if (n == 1) return;
    __threadfence();
    uint32_t p = parent_leaf[i];
    for (;;) {
        uint32_t old = atomicAdd(&flags[p], 1u);
        if (old == 0) return;
        __threadfence();
        uint32_t a = left[p], b = right[p];
        // volatile reads: the sibling's box was written by another wave
        const volatile Box* ba = (a & 0x80000000u) ? (const volatile Box*)&lbox[a & 0x7fffffffu]
                                                   : (const volatile Box*)&ibox[a];
        const volatile Box* bb = (b & 0x80000000u) ? (const volatile Box*)&lbox[b & 0x7fffffffu]
                                                   : (const volatile Box*)&ibox[b];
        Box r;
        for (int k = 0; k < 3; k++) {
            r.lo[k] = fminf(ba->lo[k], bb->lo[k]);
            r.hi[k] = fmaxf(ba->hi[k], bb->hi[k]);
        }
        ibox[p] = r;
        cnt[p] = rhi[p] - rlo[p] + 1u;
        if (R) {
            float ra[8], rb[8], out[8];
            uint8_t d[8];
            auto load = [&](uint32_t c, const volatile Box* bx, float* t) {
                const volatile float* src = R + (size_t)c * 8;
                Box q;
                for (int k = 0; k < 3; k++) {
                    q.lo[k] = bx->lo[k];
                    q.hi[k] = bx->hi[k];
                }
                for (int k = 0; k < 8; k++) t[k] = (c & 0x80000000u) ? half_area(q) * kSahTri : src[k];
            };
            load(a, ba, ra);
            load(b, bb, rb);
            sah_node(ra, rb, r, rhi[p] - rlo[p] + 1u, max_leaf, out, d);
            sah_store(R, dec, p, out, d);
        }
        __threadfence();
        if (p == 0) return;
        p = parent_int[p];
    }
}

__device__ __forceinline__ uint32_t count_of(uint32_t c, const uint32_t* cnt) {
    return (c & 0x80000000u) ? 1u : cnt[c];
}

__device__ __forceinline__ Box box_of(uint32_t c, const Box* ibox, const Box* lbox) {
    return (c & 0x80000000u) ? lbox[c & 0x7fffffffu] : ibox[c];
}

// levels a build may have: beyond kStackTotal it is refused
constexpr uint32_t kMaxLevels = (uint32_t)ltb::kStackTotal + 8u;

// One level of the BVH8.  Its nodes are slots [S_l, S_{l+1}), slot s made from
// binary node task[s]; the children of level l follow from S_{l+1} on:
// S_0 = 0, S_1 = 1, S_{k+1} = S_k + alloc[k - 1], with alloc[l] the children
// that level l allocates.  A fixed grid strides over the level, so the host
// launches levels without knowing their sizes.
__global__ __launch_bounds__(64) void k_collapse(uint32_t* __restrict__ task, uint32_t level,
                           uint32_t* __restrict__ alloc, uint32_t* __restrict__ n_tris,
                           const uint32_t* __restrict__ left, const uint32_t* __restrict__ right,
                           const uint32_t* __restrict__ cnt, const Box* __restrict__ ibox, const Box* __restrict__ lbox,
                           const uint32_t* __restrict__ sorted, const TriRec* __restrict__ tris_in,
                           TriRec* __restrict__ tris_out, Node8* __restrict__ nodes, uint32_t max_leaf,
                           const uint8_t* __restrict__ dec) {
    uint32_t s0 = 0u, s1 = 1u;
    for (uint32_t k = 0; k < level; k++) {
        s0 = s1;
        s1 += alloc[k];
    }
    for (uint32_t slot = s0 + blockIdx.x * blockDim.x + threadIdx.x; slot < s1; slot += gridDim.x * blockDim.x) {
        const uint32_t bnode = task[slot];
        uint32_t ch[8];
        int nc = 0;
        if (bnode & 0x80000000u) {
            ch[nc++] = bnode;  // a single-triangle scene
        } else if (count_of(bnode, cnt) <= max_leaf && (!dec || dec[(size_t)bnode * 8] == kDecLeaf)) {
            ch[nc++] = bnode;  // root small enough to be one leaf
        } else if (dec) {
            // the roots the SAH programme chose: the node's own split into 8,
            // then each (subtree, i roots) pair resolved by its decision
            uint32_t st_m[8], st_i[8];
            int sp = 0;
            const uint32_t k0 = dec[(size_t)bnode * 8] == kDecLeaf ? 4u : dec[(size_t)bnode * 8];
            st_m[sp] = left[bnode];
            st_i[sp++] = k0;
            st_m[sp] = right[bnode];
            st_i[sp++] = 8u - k0;
            while (sp > 0) {
                sp--;
                const uint32_t m = st_m[sp], i = st_i[sp];
                if ((m & 0x80000000u) || i == 1u) {
                    ch[nc++] = m;
                    continue;
                }
                const uint32_t dk = dec[(size_t)m * 8 + (i - 1)];
                if (dk == 0u) {
                    st_m[sp] = m;
                    st_i[sp++] = i - 1u;
                } else {
                    st_m[sp] = left[m];
                    st_i[sp++] = dk;
                    st_m[sp] = right[m];
                    st_i[sp++] = i - dk;
                }
            }
        } else {
            ch[nc++] = left[bnode];
            ch[nc++] = right[bnode];
            while (nc < 8) {
                int best = -1;
                float best_a = -1.0f;
                for (int c = 0; c < nc; c++) {
                    if (ch[c] & 0x80000000u) continue;
                    if (count_of(ch[c], cnt) <= max_leaf) continue;
                    float a = half_area(ibox[ch[c]]);
                    if (a > best_a) {
                        best_a = a;
                        best = c;
                    }
                }
                if (best < 0) break;
                uint32_t b = ch[best];
                ch[best] = left[b];
                ch[nc++] = right[b];
            }
        }
        // classify; internal children take the first slots (in their order), so
        // the traversal finds an internal child's node at child_base + slot
        uint32_t n_int = 0, n_leaf_tris = 0;
        bool is_leaf[8];
        {
            // a child is a leaf if it is a binary leaf, or holds at most max_leaf
            // triangles (and the SAH programme made it a leaf)
            auto leaf_child = [&](uint32_t c) {
                if (c & 0x80000000u) return true;
                if (count_of(c, cnt) > max_leaf) return false;
                return !dec || dec[(size_t)c * 8] == kDecLeaf || nc == 1;
            };
            uint32_t ord[8];
            int ni = 0, nl = 0;
            for (int c = 0; c < nc; c++) {
                if (leaf_child(ch[c])) {
                    n_leaf_tris += count_of(ch[c], cnt);
                } else {
                    ord[ni++] = ch[c];
                    n_int++;
                }
            }
            for (int c = 0; c < nc; c++)
                if (leaf_child(ch[c])) ord[ni + nl++] = ch[c];
            for (int c = 0; c < nc; c++) {
                ch[c] = ord[c];
                is_leaf[c] = c >= (int)n_int;
            }
        }
        const uint32_t child_base = n_int ? s1 + atomicAdd(&alloc[level], n_int) : 0u;
        const uint32_t tri_base = n_leaf_tris ? atomicAdd(n_tris, n_leaf_tris) : 0u;
        // node box and quantisation
        Box cb[8];
        Box nb;
        for (int k = 0; k < 3; k++) {
            nb.lo[k] = INFINITY;
            nb.hi[k] = -INFINITY;
        }
        for (int c = 0; c < nc; c++) {
            cb[c] = box_of(ch[c], ibox, lbox);
            for (int k = 0; k < 3; k++) {
                nb.lo[k] = fminf(nb.lo[k], cb[c].lo[k]);
                nb.hi[k] = fmaxf(nb.hi[k], cb[c].hi[k]);
            }
        }
        Node8 nd;
        int ex[3];
        for (int k = 0; k < 3; k++) {
            nd.p[k] = nb.lo[k];
            double extent = (double)nb.hi[k] - (double)nb.lo[k];
            double s = extent / 65504.0;
            int e;
            if (s <= 0.0) {
                e = -100;
            } else {
                double m = frexp(s, &e);  // s = m * 2^e, m in [0.5, 1)
                if (m == 0.5) e -= 1;
                if (ldexp(65504.0, e) < extent) e += 1;
                if (e < -100) e = -100;
            }
            ex[k] = e;
            nd.e[k] = (int8_t)e;
        }
        // internal children in the order of their centres along the longest axis
        // (the traversal's visit order): insertion sort of at most 8
        const int axis = ex[2] > max(ex[0], ex[1]) ? 2 : (ex[1] > ex[0] ? 1 : 0);
        for (int i = 1; i < (int)n_int; i++) {
            const uint32_t ci = ch[i];
            const Box bi = cb[i];
            const float key = bi.lo[axis] + bi.hi[axis];
            int j = i;
            for (; j > 0 && cb[j - 1].lo[axis] + cb[j - 1].hi[axis] > key; j--) {
                ch[j] = ch[j - 1];
                cb[j] = cb[j - 1];
            }
            ch[j] = ci;
            cb[j] = bi;
        }
        nd.imask = 0;
        nd.child_base = child_base;
        nd.tri_base = tri_base;
        uint32_t int_slot = 0, tri_off = 0;
        for (int c = 0; c < 8; c++) {
            if (c >= nc) {
                nd.meta[c] = 0;
                for (int k = 0; k < 3; k++) {
                    nd.qlo[k][c] = 0x7BFF;  // empty: lo (65504) > hi (0)
                    nd.qhi[k][c] = 0;
                }
                continue;
            }
            for (int k = 0; k < 3; k++) {
                double inv = ldexp(1.0, -ex[k]);
                nd.qlo[k][c] = f16_floor(((double)cb[c].lo[k] - (double)nd.p[k]) * inv);
                nd.qhi[k][c] = f16_ceil(((double)cb[c].hi[k] - (double)nd.p[k]) * inv);
            }
            if (is_leaf[c]) {
                // the (at most 4) triangles of the subtree, left to right
                uint32_t st[4], t = 0u;
                int sp = 0;
                st[sp++] = ch[c];
                while (sp > 0) {
                    const uint32_t m = st[--sp];
                    if (m & 0x80000000u) {
                        tris_out[tri_base + tri_off + t++] = tris_in[sorted[m & 0x7fffffffu]];
                    } else {
                        st[sp++] = right[m];
                        st[sp++] = left[m];
                    }
                }
                nd.meta[c] = (uint8_t)((tri_off << 3) | t);
                tri_off += t;
            } else {
                nd.imask |= (uint8_t)(1u << c);
                nd.meta[c] = (uint8_t)int_slot;
                task[child_base + int_slot] = ch[c];
                int_slot++;
            }
        }
        nodes[slot] = nd;
    }
}

// Structural check before any traversal runs: every internal child's index is
// larger than its parent's (so traversal terminates) and in range, and every
// leaf range lies inside the triangle array.  bad[0] = the lowest node that
// fails + 1, or 0xFFFFFFFF.
__global__ void k_check(const Node8* __restrict__ nodes, uint32_t n_nodes, uint32_t n_tris, uint32_t* __restrict__ bad) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_nodes) return;
    const Node8 nd = nodes[i];
    bool ok = true;
    for (int c = 0; c < 8; c++) {
        const uint32_t meta = nd.meta[c];
        if ((nd.imask >> c) & 1u) {
            const uint64_t ch = (uint64_t)nd.child_base + meta;
            ok = ok && ch > i && ch < n_nodes;
        } else if (meta & 7u) {
            ok = ok && (uint64_t)nd.tri_base + (meta >> 3) + (meta & 7u) <= n_tris;
        }
    }
    if (!ok) atomicMin(bad, i + 1u);
}

__global__ void k_set_u32(uint32_t* p, uint32_t n, uint32_t v) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

}  // namespace

constexpr uint32_t kMaxRounds = 200;     // PLOC rounds between two starts of their counts
constexpr uint32_t kRoundsPerSync = 8;   // rounds, levels launched between two looks at their counts
constexpr uint32_t kLevelsPerSync = 6;
// the build's counters, words of one buffer (after the six centroid bounds)
constexpr uint32_t kWMerges = 6 * kLine, kWOk = 7 * kLine, kWTris = 8 * kLine, kWBad = 9 * kLine, kWRounds = 10 * kLine,
                   kWLevels = kWRounds + kMaxRounds + 1, kBuildWords = kWLevels + kMaxLevels;
constexpr size_t kBuildKeepBytes = 512ull << 20;

lt_status bvh_build(lt_context* ctx, const lt_build_opts* opts, lt_build_stats* stats) {
    if (!ctx->scene.uploaded) return lt_fail(ctx, LT_ERR_NOT_READY, "lt_accel_build: no scene uploaded");
    uint32_t max_leaf = opts && opts->max_leaf_tris ? opts->max_leaf_tris : 1u;
    if (max_leaf < 1 || max_leaf > 4) return lt_fail(ctx, LT_ERR_INVALID_ARG, "max_leaf_tris must be in 1..4");
    const uint32_t collapse = opts && opts->collapse ? opts->collapse : LT_COLLAPSE_SAH;
    if (collapse != LT_COLLAPSE_SAH && collapse != LT_COLLAPSE_GREEDY)
        return lt_fail(ctx, LT_ERR_INVALID_ARG, "unknown collapse");
    const bool sah = collapse == LT_COLLAPSE_SAH;
    const uint32_t tree = opts && opts->binary_tree ? opts->binary_tree : LT_TREE_PLOC;
    if (tree != LT_TREE_PLOC && tree != LT_TREE_LBVH) return lt_fail(ctx, LT_ERR_INVALID_ARG, "unknown binary tree");
    hipStream_t st = ctx->stream;
    DeviceBVH& bvh = ctx->bvh;
    if (bvh.nodes) (void)hipFree(bvh.nodes);
    if (bvh.tris) (void)hipFree(bvh.tris);
    bvh = DeviceBVH{};
    const uint32_t n = ctx->scene.ntris;
    LT_HIP(ctx, hipEventRecord(ctx->ev0, st));
    if (n == 0) {
        bvh.built = true;
        if (stats) *stats = lt_build_stats{};
        return LT_OK;
    }
    const bool ploc = tree == LT_TREE_PLOC;
    const uint32_t ni = n > 1 ? n - 1 : 1;
    const int B = 256;
    const uint32_t G = (n + B - 1) / B;
    size_t sort_bytes = 0;
    LT_HIP(ctx, rocprim::radix_sort_pairs(nullptr, sort_bytes, (uint32_t*)nullptr, (uint32_t*)nullptr,
                                          (uint32_t*)nullptr, (uint32_t*)nullptr, n, 0u, 30u, st));
    // One workspace for every temporary, laid out twice: first for its size,
    // then over its memory.  The context keeps it for the next build up to
    // kBuildKeepBytes (allocating and freeing 45 buffers took 3 ms of a
    // 12 ms build of 250k triangles).
    TriRec* tris_unsorted;
    uint32_t *words, *keys, *vals, *keys2, *vals2, *left, *right, *cnt, *task;
    Box *ibox, *lbox;
    Node8* nodes;
    float* sah_R;
    uint8_t* sah_dec;
    void* sort_tmp;
    uint32_t *cl_node0 = nullptr, *cl_node1 = nullptr, *kept = nullptr;
    Box *cl_box0 = nullptr, *cl_box1 = nullptr;
    uint32_t *pint = nullptr, *pleaf = nullptr, *rlo = nullptr, *rhi = nullptr, *flags = nullptr;
    size_t bytes = 0;
    char* mem = nullptr;
    auto take = [&](auto*& p, size_t count) {
        using T = std::remove_reference_t<decltype(*p)>;
        p = (T*)(mem ? mem + bytes : nullptr);
        bytes += (count * sizeof(T) + 255) / 256 * 256;
    };
    auto layout = [&]() {
        bytes = 0;
        take(words, kBuildWords);
        take(tris_unsorted, n);
        take(nodes, n);
        take(keys, n);
        take(vals, n);
        take(keys2, n);
        take(vals2, n);
        take(left, ni);
        take(right, ni);
        take(cnt, ni);
        take(task, n);
        take(ibox, ni);
        take(lbox, n);
        take(sah_R, sah ? (size_t)8 * ni : 0);
        take(sah_dec, sah ? (size_t)8 * ni : 0);
        char* tmp;
        take(tmp, sort_bytes);
        sort_tmp = tmp;
        if (ploc) {
            take(cl_node0, n);
            take(cl_node1, n);
            take(cl_box0, n);
            take(cl_box1, n);
            take(kept, (n + kPlocBlock - 1) / kPlocBlock);
        } else {
            take(pint, ni);
            take(pleaf, n);
            take(rlo, ni);
            take(rhi, ni);
            take(flags, ni);
        }
    };
    layout();
    if (ctx->build_ws_bytes < bytes) {
        if (ctx->build_ws) (void)hipFree(ctx->build_ws);
        ctx->build_ws = nullptr;
        ctx->build_ws_bytes = 0;
        LT_HIP(ctx, hipMalloc(&ctx->build_ws, bytes));
        ctx->build_ws_bytes = bytes;
    }
    mem = (char*)ctx->build_ws;
    layout();
    // words: centroid bounds, merges, PLOC progress flag, leaf triangles, the
    // check's verdict, then m per PLOC round, alloc per level
    uint32_t *cb = words, *mctr = words + kWMerges, *ok = words + kWOk, *n_tris = words + kWTris, *bad = words + kWBad,
             *m_of = words + kWRounds, *alloc = words + kWLevels;
    lt_status rc = LT_OK;
    auto build = [&]() -> lt_status {
        uint32_t h_words[kBuildWords] = {};
        for (int k = 0; k < 3; k++) h_words[k * kLine] = 0xFFFFFFFFu;  // minima
        h_words[kWOk] = 1u;
        h_words[kWBad] = 0xFFFFFFFFu;
        h_words[kWRounds] = n;
        LT_HIP(ctx, hipMemcpyAsync(words, h_words, sizeof(h_words), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(k_make_tris, dim3(std::min(G, 2u * (uint32_t)ctx->num_cus)), dim3(B), 0, st, ctx->scene.vtx, ctx->scene.idx, ctx->scene.prims,
                           ctx->scene.tri_start, ctx->scene.xf, ctx->scene.nprims, n, tris_unsorted, cb);
        hipLaunchKernelGGL(k_morton, dim3(G), dim3(B), 0, st, tris_unsorted, n, cb, keys, vals);
        LT_HIP(ctx, hipGetLastError());
        LT_HIP(ctx, rocprim::radix_sort_pairs(sort_tmp, sort_bytes, keys, keys2, vals, vals2, n, 0u, 30u, st));
        if (ploc) {
            const PlocTree T{left, right, cnt, ibox, lbox, sah ? sah_R : nullptr, sah_dec, n, max_leaf};
            hipLaunchKernelGGL(k_ploc_init, dim3(G), dim3(B), 0, st, tris_unsorted, vals2, n, cl_node0, cl_box0, lbox);
            uint32_t m = n, round = 0;
            while (m > kPlocTail) {
                // rounds shrink the clusters by about a third: a few at a time on the grid of the first
                const uint32_t gm = (m + kPlocBlock - 1) / kPlocBlock, last = std::min(round + kRoundsPerSync, kMaxRounds);
                for (; round < last; round++) {
                    hipLaunchKernelGGL(k_ploc_merge, dim3(gm), dim3(kPlocBlock), 0, st, T, cl_node0, cl_box0, m_of, round,
                                       mctr, cl_node1, cl_box1, kept);
                    hipLaunchKernelGGL(k_ploc_compact, dim3(gm), dim3(kPlocBlock), 0, st, cl_node1, cl_box1, m_of, round,
                                       kept, cl_node0, cl_box0);
                }
                LT_HIP(ctx, hipGetLastError());
                uint32_t m_next;
                LT_HIP(ctx, hipMemcpyAsync(&m_next, m_of + round, 4, hipMemcpyDeviceToHost, st));
                LT_HIP(ctx, hipStreamSynchronize(st));
                if (m_next >= m) return lt_fail(ctx, LT_ERR_HIP, "PLOC round merged no clusters");
                m = m_next;
                if (round == kMaxRounds) {  // slow merging: the counts start over
                    round = 0;
                    hipLaunchKernelGGL(k_set_u32, dim3(1), dim3(64), 0, st, m_of, 1u, m);
                }
            }
            if (n > 1)
                hipLaunchKernelGGL(k_ploc_tail, dim3(1), dim3(kTailBlock), 0, st, T, cl_node0, cl_box0, m_of, round, mctr, ok);
            LT_HIP(ctx, hipGetLastError());
        } else {
            if (n > 1)
                hipLaunchKernelGGL(k_karras, dim3((n - 1 + B - 1) / B), dim3(B), 0, st, keys2, (int)n, left, right, pint,
                                   pleaf, rlo, rhi);
            hipLaunchKernelGGL(k_set_u32, dim3((ni + B - 1) / B), dim3(B), 0, st, flags, ni, 0u);
            hipLaunchKernelGGL(k_refit, dim3(G), dim3(B), 0, st, tris_unsorted, vals2, (int)n, left, right, pint, pleaf,
                               flags, ibox, lbox, rlo, rhi, max_leaf, sah ? sah_R : nullptr, sah_dec, cnt);
            LT_HIP(ctx, hipGetLastError());
        }
        LT_HIP(ctx, hipMalloc(&bvh.tris, sizeof(TriRec) * n));
        // top-down collapse, one launch per BVH8 level, a few levels between
        // two looks at what they allocated
        hipLaunchKernelGGL(k_set_u32, dim3(1), dim3(64), 0, st, task, 1u, n > 1 ? 0u : 0x80000000u);
        const uint32_t grid = std::min<uint32_t>((n + 63) / 64, 4096u);
        uint32_t level = 0, depth = 0;
        while (depth == 0) {
            if (level >= kMaxLevels)
                return lt_fail(ctx, LT_ERR_UNSUPPORTED, "BVH8 depth exceeds the traversal stack bound of " +
                                                            std::to_string(ltb::kStackTotal));
            const uint32_t first = level;
            for (; level < std::min(first + kLevelsPerSync, kMaxLevels); level++)
                hipLaunchKernelGGL(k_collapse, dim3(grid), dim3(64), 0, st, task, level, alloc, n_tris, left, right, cnt,
                                   ibox, lbox, vals2, tris_unsorted, bvh.tris, nodes, max_leaf, sah ? sah_dec : nullptr);
            LT_HIP(ctx, hipGetLastError());
            LT_HIP(ctx, hipMemcpyAsync(h_words, words, sizeof(h_words), hipMemcpyDeviceToHost, st));
            LT_HIP(ctx, hipStreamSynchronize(st));
            if (h_words[kWOk] == 0u) return lt_fail(ctx, LT_ERR_HIP, "PLOC round merged no clusters");
            for (uint32_t l = first; l < level && depth == 0; l++)
                if (h_words[kWLevels + l] == 0u) depth = l + 1;
        }
        uint32_t n_nodes = 1;
        for (uint32_t l = 0; l < depth; l++) n_nodes += h_words[kWLevels + l];
        bvh.n_nodes = n_nodes;
        bvh.n_tris = h_words[kWTris];
        bvh.depth = depth;
        if (bvh.n_tris != n) return lt_fail(ctx, LT_ERR_HIP, "BVH collapse lost triangles");
        // traversal stack: one group entry per ancestor level; entries pack
        // child_base << 8, so node indices must stay below 2^24
        if (depth > (uint32_t)ltb::kStackTotal)
            return lt_fail(ctx, LT_ERR_UNSUPPORTED,
                           "BVH8 depth " + std::to_string(depth) + " exceeds the traversal stack bound");
        if (bvh.n_nodes >= (1u << 24)) return lt_fail(ctx, LT_ERR_UNSUPPORTED, "BVH8 has more than 2^24 nodes");
        LT_HIP(ctx, hipMalloc(&bvh.nodes, sizeof(Node8) * (size_t)n_nodes));
        LT_HIP(ctx, hipMemcpyAsync(bvh.nodes, nodes, sizeof(Node8) * (size_t)n_nodes, hipMemcpyDeviceToDevice, st));
        hipLaunchKernelGGL(k_check, dim3((n_nodes + B - 1) / B), dim3(B), 0, st, bvh.nodes, n_nodes, n, bad);
        LT_HIP(ctx, hipGetLastError());
        LT_HIP(ctx, hipEventRecord(ctx->ev1, st));
        Node8 root;
        uint32_t verdict = 0;
        LT_HIP(ctx, hipMemcpyAsync(&root, bvh.nodes, sizeof(root), hipMemcpyDeviceToHost, st));
        LT_HIP(ctx, hipMemcpyAsync(&verdict, bad, 4, hipMemcpyDeviceToHost, st));
        LT_HIP(ctx, hipStreamSynchronize(st));
        if (verdict != 0xFFFFFFFFu)
            return lt_fail(ctx, LT_ERR_HIP, "BVH8 node " + std::to_string(verdict - 1u) + " has a bad child or leaf");
        for (int k = 0; k < 3; k++) {
            // non-negative fp16 bit patterns are ordered as their values; an empty slot's is 0
            const uint16_t q = *std::max_element(root.qhi[k], root.qhi[k] + 8);
            bvh.root_lo[k] = root.p[k];
            bvh.root_hi[k] = root.p[k] + std::ldexp((float)__builtin_bit_cast(_Float16, q), root.e[k]);
        }
        float ms = 0.0f;
        LT_HIP(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        bvh.built = true;
        if (stats) {
            stats->num_nodes = bvh.n_nodes;
            stats->num_tris = bvh.n_tris;
            stats->max_depth = depth;
            stats->binary_depth = 0;
            stats->build_ms = ms;
        }
        return LT_OK;
    };
    rc = build();
    if (rc != LT_OK) {
        (void)hipStreamSynchronize(st);
        if (bvh.nodes) (void)hipFree(bvh.nodes);
        if (bvh.tris) (void)hipFree(bvh.tris);
        bvh = DeviceBVH{};
    }
    if (ctx->build_ws_bytes > kBuildKeepBytes) {
        (void)hipFree(ctx->build_ws);
        ctx->build_ws = nullptr;
        ctx->build_ws_bytes = 0;
    }
    return rc;
}
