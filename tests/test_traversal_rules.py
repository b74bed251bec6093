"""Rules of the BVH8 traversal that need no GPU, through the host replay of the
device's node walk (oracle/oracle_bvh8.cpp, same bounds and child order) over
a BVH8 made on the host."""
import numpy as np
import pytest

import host_bvh8
import lumen_amd as la
import oracle
from lumen_amd._abi import RAY_DTYPE

from raygen import aimed_rays, random_rays


def _soup(n, seed, size=0.1):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-2, 2, (n, 1, 3)) + rng.uniform(-size, size, (n, 3, 3))).astype(np.float32)


def bad_rays(tri):
    """Rays that cannot hit anything: a NaN in one or all components of the
    origin or the direction, and an empty interval."""
    base = np.concatenate([random_rays(tri, 16, 1), aimed_rays(tri, 16, 2)])
    out = []
    for field in ("org", "dir"):
        for k in (0, 1, 2, slice(None)):
            for sign in (1.0, -1.0):
                r = base.copy()
                r[field][:, k] = np.copysign(np.float32(np.nan), np.float32(sign))
                out.append(r)
    r = base.copy()
    r["tmax"] = -1e4
    out.append(r)
    return np.concatenate(out).astype(RAY_DTYPE)


@pytest.mark.parametrize("any_hit", [False, True])
def test_rays_that_cannot_hit_visit_at_most_the_root(any_hit):
    tri = _soup(3000, 3)
    nodes, tris = host_bvh8.build(tri)
    good = np.concatenate([random_rays(tri, 200, 4), aimed_rays(tri, 200, 5)])
    hits, nc, _ = oracle.bvh8_trace(nodes, tris, good, any_hit)
    assert (hits if any_hit else hits["inst"] != 0xFFFFFFFF).any() and nc.min() >= 1
    rays = bad_rays(tri)
    hits, nc, tc = oracle.bvh8_trace(nodes, tris, rays, any_hit)
    assert not (hits if any_hit else hits["inst"] != 0xFFFFFFFF).any()
    assert nc.max() <= 1 and tc.max() == 0, (nc.max(), tc.max())


@pytest.mark.parametrize("scale", [1.0, 37.0, 2.0 ** -20])
def test_the_surfaces_at_a_rays_ends_are_not_tested(scale):
    """The cull margin is 2^-16 of the farthest point of the scene along the ray's
    dominant axis (and the slab error 2^-20 of the extent): segments between two
    walls of a box of extent 1 that keep 2^-15 from both test no triangle."""
    from scenes import box_faces
    tri = np.concatenate([np.array(f, np.float32) for f in box_faces((0, 0, 0), (1, 1, 1))])
    tri *= np.float32(scale)
    nodes, tris = host_bvh8.build(tri)
    rng = np.random.default_rng(2)
    n = 600
    r = np.zeros(n, RAY_DTYPE)
    ax, up = rng.integers(0, 3, n), rng.random(n) < 0.5
    o, d = rng.uniform(0.3, 0.7, (n, 3)), rng.uniform(-0.2, 0.2, (n, 3))
    i = np.arange(n)
    gap = 2.0 ** -15
    o[i, ax] = np.where(up, gap, 1 - gap)
    d[i, ax] = np.where(up, 1.0, -1.0)
    r["org"], r["dir"], r["tmin"], r["tmax"] = o * scale, d, 0.0, (1 - 2 * gap) * scale
    occ, nc, tc = oracle.bvh8_trace(nodes, tris, r, True)
    assert not occ.any() and nc.min() >= 1
    assert tc.sum() == 0, tc.mean()


@pytest.mark.gpu
@pytest.mark.parametrize("any_hit", [False, True])
def test_rays_that_cannot_hit_on_the_device(gpu_ctx, any_hit):
    print(f"[gpu] rays that cannot hit, any={any_hit}", flush=True)
    sc = la.Scene.procedural("terrain", seed=2, terrain_tris=5000)
    gpu_ctx.upload(sc)
    gpu_ctx.build_accel()
    rays = bad_rays(sc.triangles())
    got = gpu_ctx.trace_any(rays) if any_hit else gpu_ctx.trace_closest(rays)["inst"] != 0xFFFFFFFF
    assert not got.any()
    nodes, tris = gpu_ctx.trace_count(rays, any_hit)
    assert nodes <= len(rays) and tris == 0, (nodes, tris)
    nan = np.concatenate([rays[:64], rays[:64]])  # a NaN limit: no hit either
    nan["org"], nan["dir"] = random_rays(sc.triangles(), 128, 7)["org"], random_rays(sc.triangles(), 128, 7)["dir"]
    nan["tmin"][:64], nan["tmax"][64:] = np.nan, np.nan
    got = gpu_ctx.trace_any(nan) if any_hit else gpu_ctx.trace_closest(nan)["inst"] != 0xFFFFFFFF
    assert not got.any()
