"""Edges of the BVH8 traversal: leaves of 1 to 4 triangles (the triangle masks
of a leaf group), rays that run exactly along an axis or a node's plane, far
origins (the per-ray rounding bounds), unnormalised directions, and a tree
deeper than the LDS stack.  Hits are bit-identical to brute force: the
traversal may only visit more, never miss."""
import numpy as np
import pytest

import lumen_amd as la
import oracle
from raygen import aimed_rays, random_rays
from scenes import DescScene

pytestmark = pytest.mark.gpu


def _upload(ctx, desc, max_leaf=1):
    sc = la.Scene.__new__(la.Scene)
    sc._h = None
    sc.desc = desc
    ctx.upload(sc)
    return sc, ctx.build_accel(max_leaf)


def _same(ctx, desc, rays, tag):
    acc = oracle.Accel(desc)
    g, o = ctx.trace_closest(rays), acc.closest(rays, brute=True)
    for f in ("inst", "prim"):
        assert np.array_equal(g[f], o[f]), f"{tag}: {f}"
    for f in ("t", "u", "v"):
        assert np.array_equal(g[f].view(np.uint32), o[f].view(np.uint32)), f"{tag}: {f}"
    assert np.array_equal(ctx.trace_any(rays), acc.any(rays, brute=True)), f"{tag}: any"
    return g


def _soup(n, seed, size=0.3):
    rng = np.random.default_rng(seed)
    s = DescScene()
    m = s.material(bsdf_type=1, bsdf_props=9, albedo=(0.5, 0.5, 0.5))
    c = rng.uniform(-2, 2, (n, 1, 3))
    s.mesh((c + rng.uniform(-size, size, (n, 3, 3))).astype(np.float32), m)
    return s


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 40, 700])
@pytest.mark.parametrize("max_leaf", [1, 2, 3, 4])
def test_leaf_groups(gpu_ctx, n, max_leaf):
    print(f"[gpu] leaf groups n={n} max_leaf={max_leaf}", flush=True)
    s = _soup(n, 100 + n)
    d = s.build()
    sc, st = _upload(gpu_ctx, d, max_leaf)
    assert st.num_tris == n
    t = sc.triangles()
    _same(gpu_ctx, d, np.concatenate([random_rays(t, 700, 1), aimed_rays(t, 700, 2)]), f"n={n}")


@pytest.mark.parametrize("kind", ["axis", "far", "scaled", "planar"])
def test_ray_edges(gpu_ctx, kind):
    print(f"[gpu] ray edges {kind}", flush=True)
    rng = np.random.default_rng(7)
    s = _soup(300, 5)
    m = 0
    if kind == "planar":  # axis-aligned walls and duplicates: nodes without extent on an axis
        s = DescScene()
        m = s.material(bsdf_type=1, bsdf_props=9, albedo=(0.5, 0.5, 0.5))
        g = np.array([[x, y] for x in range(6) for y in range(6)], np.float32)
        for ax in range(3):
            q = np.zeros((36, 3, 3), np.float32)
            for k, (du, dv) in enumerate(((0, 0), (1, 0), (0, 1))):
                q[:, k, (ax + 1) % 3], q[:, k, (ax + 2) % 3] = g[:, 0] + du, g[:, 1] + dv
            s.mesh(np.concatenate([q, q[:5], np.repeat(q[:1, :1], 3, 1)]), m)  # + duplicates, a point
    d = s.build()
    sc, _ = _upload(gpu_ctx, d)
    t = sc.triangles()
    lo, hi = t.reshape(-1, 3).min(0), t.reshape(-1, 3).max(0)
    n = 1500
    rays = np.concatenate([random_rays(t, n, 3), aimed_rays(t, n, 4)])
    if kind in ("axis", "planar"):
        a = np.concatenate([random_rays(t, n, 5), aimed_rays(t, n, 6)])
        dirs = np.zeros((len(a), 3), np.float32)
        dirs[np.arange(len(a)), rng.integers(0, 3, len(a))] = rng.choice([-1.0, 1.0], len(a))
        dirs[::3, 0] += np.float32(1e-20)  # nearly parallel
        a["dir"] = dirs
        a["org"][: n // 2] = t.reshape(-1, 3)[rng.integers(0, 3 * len(t), n // 2)]  # on vertices
        rays = np.concatenate([rays, a])
    if kind == "far":
        rays["org"] = (lo + hi) / 2 + (rays["org"] - (lo + hi) / 2) * np.float32(3e4)
        tgt = t.mean(1)[rng.integers(0, len(t), len(rays))]
        rays["dir"] = tgt - rays["org"]
    if kind == "scaled":
        rays["dir"] *= np.exp(rng.uniform(-18, 18, (len(rays), 1))).astype(np.float32)
    g = _same(gpu_ctx, d, rays, kind)
    assert (g["inst"] != 0xFFFFFFFF).any()


def test_tree_deeper_than_the_lds_stack(gpu_ctx):
    """Triangles whose sizes and distances from the origin halve: a chain-like
    tree, more levels than the 16 LDS entries serve, entered from the far end
    so that groups wait on every level."""
    print("[gpu] deep tree", flush=True)
    s = DescScene()
    m = s.material(bsdf_type=1, bsdf_props=9, albedo=(0.5, 0.5, 0.5))
    k = 2.0 ** (-0.5 * np.arange(220))
    base = np.array([[1, 0.2, 0], [1.2, -0.2, 0.1], [1.1, 0, 0.3]])
    s.mesh((k[:, None, None] * base).astype(np.float32), m)
    d = s.build()
    sc, st = _upload(gpu_ctx, d)
    print(f"[gpu] depth {st.max_depth}", flush=True)
    assert st.max_depth > 17
    t = sc.triangles()
    rays = np.concatenate([random_rays(t, 2000, 8), aimed_rays(t, 4000, 9)])
    c = t.mean(1)[np.random.default_rng(1).integers(0, len(t), 4000)]
    r = aimed_rays(t, 4000, 10)
    r["org"] = np.array([0, 0, 0], np.float32)
    r["dir"] = c * np.float32(1e6)
    _same(gpu_ctx, d, np.concatenate([rays, r]), "deep")
