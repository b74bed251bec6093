"""The BVH build around the sizes where its steps change: one triangle, a
PLOC workgroup and its halo, the cluster count at which one workgroup takes
the remaining rounds, several workgroups; both binary trees and collapses; a
workspace reused by builds of other sizes; a chain too deep for the traversal
stack.  Hits are bit-identical to brute force, and PLOC's tree does not
depend on how its rounds are launched."""
import numpy as np
import pytest

import lumen_amd as la
import oracle
from raygen import aimed_rays, random_rays
from scenes import DescScene

pytestmark = pytest.mark.gpu


def _scene(n, seed, clustered=False):
    rng = np.random.default_rng(seed)
    s = DescScene()
    m = s.material(bsdf_type=1, bsdf_props=9, albedo=(0.5, 0.5, 0.5))
    c = rng.normal(size=(n, 1, 3)) if clustered else rng.uniform(-2, 2, (n, 1, 3))
    s.mesh((c + rng.uniform(-0.1, 0.1, (n, 3, 3))).astype(np.float32), m)
    d = s.build()
    sc = la.Scene.__new__(la.Scene)
    sc._h = None
    sc.desc = d
    sc._keep = s
    return sc


@pytest.mark.parametrize("tree,collapse", [("ploc", "sah"), ("ploc", "greedy"), ("lbvh", "sah")])
def test_builds_of_every_size_class(gpu_ctx, tree, collapse):
    for n in (1, 2, 3, 31, 255, 256, 257, 300, 2047, 2048, 2049, 2305, 5000):  # down and up again: the workspace
        for k in (n, 7) if n == 5000 else (n,):
            print(f"[gpu] build {tree} {collapse} n={k}", flush=True)
            sc = _scene(k, k, clustered=k % 2 == 0)
            gpu_ctx.upload(sc)
            st = gpu_ctx.build_accel(1 + k % 4, collapse=collapse, tree=tree)
            assert st.num_tris == k
            nodes, tris = gpu_ctx.export_bvh(st)
            gid = np.sort(tris[:, 36:40].copy().view(np.uint32)[:, 0])
            assert np.array_equal(gid, np.arange(k))  # every triangle once
            t = sc.triangles()
            rays = np.concatenate([random_rays(t, 300, 1), aimed_rays(t, 300, 2)])
            acc = oracle.Accel(sc.desc)
            g, o = gpu_ctx.trace_closest(rays), acc.closest(rays, brute=True)
            assert np.array_equal(g.view(np.uint8), o.view(np.uint8)), (tree, collapse, k)


def _nested(n):
    """n triangles whose boxes are nested cubes, the smallest first.  A union's
    box is the larger one's, so of all pairs only the two smallest clusters
    prefer each other: PLOC merges one pair a round into a chain of n - 1
    nodes, and a BVH8 node takes 7 of its triangles and the rest, whichever
    collapse: (n - 1) / 7 levels."""
    s = DescScene()
    m = s.material(bsdf_type=1, bsdf_props=9, albedo=(0.5, 0.5, 0.5))
    k = np.exp2(np.linspace(-72, 20, n))
    base = np.array([[-1, -1, -1], [1, 1, -1], [1, -1, 1]])
    s.mesh((k[:, None, None] * base).astype(np.float32), m, normals=np.tile(np.float32([0, 0, 1]), (n, 3, 1)))
    sc = la.Scene.__new__(la.Scene)
    sc._h = None
    sc.desc = s.build()
    sc._keep = s
    return sc


# 1370: 193..200 levels, found after the last level; 2000: more levels than are
# launched at all; 2600: also PLOC rounds beyond one start of their counts
@pytest.mark.parametrize("collapse", ["sah", "greedy"])
@pytest.mark.parametrize("n", [1370, 2000, 2600])
def test_a_chain_too_deep_is_refused(gpu_ctx, n, collapse):
    print(f"[gpu] too deep a chain {n} {collapse}", flush=True)
    gpu_ctx.upload(_nested(n))
    with pytest.raises(la.LtError, match="stack bound"):
        gpu_ctx.build_accel(collapse=collapse)
    ok = _scene(50, 1)  # the context stays usable
    gpu_ctx.upload(ok)
    assert gpu_ctx.build_accel().num_tris == 50
    t = ok.triangles()
    rays = np.concatenate([random_rays(t, 300, 1), aimed_rays(t, 300, 2)])
    g, o = gpu_ctx.trace_closest(rays), oracle.Accel(ok.desc).closest(rays, brute=True)
    assert np.array_equal(g.view(np.uint8), o.view(np.uint8))


def test_the_deepest_chain_is_traced(gpu_ctx):
    print("[gpu] deepest chain", flush=True)
    sc = _nested(1340)
    gpu_ctx.upload(sc)
    st = gpu_ctx.build_accel()
    assert 185 <= st.max_depth <= 192, st.max_depth
    t = sc.triangles()
    rays = np.concatenate([random_rays(t[-200:], 1000, 1), aimed_rays(t[-200:], 1000, 2), aimed_rays(t[600:], 1000, 3)])
    g, o = gpu_ctx.trace_closest(rays), oracle.Accel(sc.desc).closest(rays, brute=True)
    assert (g["inst"] != 0xFFFFFFFF).any()
    assert np.array_equal(g.view(np.uint8), o.view(np.uint8))
