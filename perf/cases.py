"""The framework's workloads as measurable cases: raw ray queries, scene
(re)builds, the four integrators and the texture adjoint, each through the
public entry points that a user's program calls.

A case is a dict of plain values.  ``prepare`` makes what a program holds
before the call (scene on the GPU, BVH, integrator, rays or texels), ``run``
is one pass, ``exact`` the same outputs from plain torch in 64 bits where a
brute-force evaluation is affordable.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import lumen_amd as la
from lumen_amd import _abi
from lumen_amd.adjoint import Adjoint, render_textures


# ------------------------------------------------------------------ cases ----
def listed():
    return [
        # picking and visibility probes of an interactive host: a few rays, latency only
        dict(name="closest_cornell_1k", kind="trace", scene="cornell", tris=36, n=1023, any=False, rays="mixed"),
        # a host renderer's incoherent bounce rays over a large scene
        dict(name="closest_terrain_2m", kind="trace", scene="terrain", tris=1000000, n=2073600, any=False,
             rays="bounce"),
        # its shadow rays, an odd count over a middle-sized scene
        dict(name="any_terrain_333k", kind="trace", scene="terrain", tris=250000, n=333331, any=True, rays="shadow"),
        # an animated scene: new geometry uploaded, the BVH rebuilt, one batch of queries
        dict(name="rebuild_terrain_250k", kind="rebuild", scene="terrain", tris=250000, n=65536, rays="bounce"),
        # the headline workload: 1080p Path frames of the 1M-triangle terrain, accumulated and read back
        dict(name="path_terrain_1080p", kind="path", scene="terrain", tris=1000000, width=1920, height=1080, depth=12,
             spp=16, strategy="persistent"),
        # the integrator's default strategy on the Cornell box, odd image size
        dict(name="path_cornell_509", kind="path", scene="cornell", tris=36, width=509, height=383, depth=6, spp=16,
             strategy="megakernel"),
        # an interactive preview: one sample per pixel of a small window
        dict(name="path_preview_160", kind="path", scene="caustics", tris=20000, width=160, height=120, depth=8, spp=1,
             strategy="megakernel"),
        # bidirectional frames of the caustics scene
        dict(name="bdpt_caustics_1024", kind="bdpt", scene="caustics", tris=20000, width=1024, height=1024, depth=8,
             spp=8, mis="power"),
        # vertex connection and merging over 1,048,576 light paths a frame
        dict(name="vcm_caustics_1024", kind="vcm", scene="caustics", tris=20000, width=1024, height=1024, depth=8,
             spp=8, estimator="corrected", vm=True, radius=1.0, alpha=0.75),
        # the default (reference) VCM estimator at a window's size
        dict(name="vcm_reference_501", kind="vcm", scene="caustics", tris=20000, width=501, height=377, depth=6,
             spp=4, estimator="reference", vm=True, radius=0.5, alpha=0.75),
        # progressive photon mapping frames
        dict(name="sppm_caustics_1024", kind="sppm", scene="caustics", tris=20000, width=1024, height=1024, depth=8,
             spp=8, radius=0.03),
        # inverse rendering: forward and backward of 32 texture variants (quarter of the samples of the
        # 512 x 512, 32-sample benchmark)
        dict(name="adjoint_wall_512", kind="adjoint", scene="diff_wall", tris=16384, tex=256, width=512, height=512,
             depth=6, spp=8, variants=32, cache=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "trace", "rebuild", "path", "path", "bdpt", "vcm", "sppm", "adjoint"])
    scene = rng.choice(["terrain", "caustics", "cornell"])
    tris = {"terrain": _log(rng, 2000, 1000000), "caustics": _log(rng, 500, 100000), "cornell": 36}[scene]
    w = _log(rng, 96, 1440)
    h = max(64, min(1080, int(w * rng.uniform(0.5, 1.0))))
    spp = max(1, min(16, int(rng.uniform(0.3, 1.0) * 8e6 / (w * h))))
    if kind == "trace":
        any_hit = rng.random() < 0.4
        return dict(kind=kind, scene=scene, tris=tris, n=_log(rng, 500, 2000000), any=any_hit,
                    rays="shadow" if any_hit else rng.choice(["bounce", "camera", "mixed"]))
    if kind == "rebuild":
        return dict(kind=kind, scene=rng.choice(["terrain", "caustics"]), tris=_log(rng, 2000, 250000),
                    n=_log(rng, 1000, 65536), rays="bounce")
    if kind == "path":
        return dict(kind=kind, scene=scene, tris=tris, width=w, height=h, depth=rng.randint(2, 12), spp=spp,
                    strategy=rng.choice(["persistent", "megakernel", "wavefront"]))
    # the bidirectional integrators on the scenes they are used for
    scene = rng.choice(["caustics", "cornell"])
    tris = _log(rng, 500, 50000) if scene == "caustics" else 36
    w, h = min(w, 1024), min(h, 800)
    spp = max(1, spp // 2)
    if kind == "bdpt":
        return dict(kind=kind, scene=scene, tris=tris, width=w, height=h, depth=rng.randint(2, 8), spp=spp,
                    mis=rng.choice(["balance", "power"]))
    if kind == "vcm":
        return dict(kind=kind, scene=scene, tris=tris, width=w, height=h, depth=rng.randint(2, 8), spp=spp,
                    estimator=rng.choice(["corrected", "reference"]), vm=rng.random() < 0.8,
                    radius=rng.uniform(0.2, 1.0), alpha=0.75)
    if kind == "sppm":
        return dict(kind=kind, scene=scene, tris=tris, width=w, height=h, depth=rng.randint(2, 8), spp=spp,
                    radius=rng.uniform(0.01, 0.04))
    w = _log(rng, 48, 256)
    return dict(kind="adjoint", scene="diff_wall", tris=_log(rng, 200, 16384), tex=rng.choice([32, 100, 256]),
                width=w, height=max(40, int(w * rng.uniform(0.6, 1.0))), depth=rng.randint(2, 7),
                spp=rng.randint(1, 16), variants=rng.choice([1, 3, 8, 32]), cache=rng.random() < 0.8)


# ----------------------------------------------------------------- inputs ----
def _scene(case, seed):
    key = {"terrain": "terrain_tris", "caustics": "sphere_tris", "diff_wall": "wall_tris"}.get(case["scene"])
    kw = {key: case["tris"]} if key else {}
    if case["scene"] == "diff_wall":
        kw["tex_res"] = case["tex"]
    return la.Scene.procedural(case["scene"], seed=1 + seed % 1000003, **kw)


def _camera_dirs(cam, x, y, w, h):
    """Camera-space unit directions through pixel positions (x, y), as world rays."""
    inv_v = torch.tensor(list(cam.inv_view), device=x.device).view(4, 4).T
    inv_p = torch.tensor(list(cam.inv_projection), device=x.device).view(4, 4).T
    ndc = torch.stack([2 * x / w - 1, 2 * y / h - 1, torch.ones_like(x), torch.ones_like(x)], 1)
    d = torch.nn.functional.normalize((ndc @ inv_p.T)[:, :3], dim=1) @ inv_v[:3, :3].T
    return inv_v[:3, 3].expand_as(d), d


def _rays(case, scene, seed, rays=None):
    """[n, 8] float32 rays (origin, tmin, direction, tmax) as renderers cast them:
    camera rays in scanline order, cosine-distributed bounces off surface
    points, or segments from surface points towards a light."""
    n, g = case["n"], torch.Generator("cuda").manual_seed(seed)
    rays = rays or case["rays"]
    if rays == "mixed":
        m = dict(case, n=(n + 1) // 2), dict(case, n=n // 2)
        return torch.cat([_rays(m[0], scene, seed, "camera"), _rays(m[1], scene, seed + 1, "bounce")])
    out = torch.empty(n, 8, device="cuda")
    out[:, 3], out[:, 7] = 0.001, 1e4
    rnd = lambda *s: torch.rand(*s, generator=g, device="cuda")
    if rays == "camera":
        w = max(1, int(math.sqrt(n * 16 / 9)))
        h = -(-n // w)
        i = torch.arange(n, device="cuda")
        o, d = _camera_dirs(scene.camera(w, h), i % w + rnd(n), torch.div(i, w, rounding_mode="floor") + rnd(n), w, h)
    else:
        tri = torch.from_numpy(scene.triangles()).cuda()
        t = tri[torch.randint(len(tri), (n,), generator=g, device="cuda")]
        s, b = rnd(n, 1).sqrt(), rnd(n, 1)
        p = t[:, 0] * (1 - s) + t[:, 1] * (s * (1 - b)) + t[:, 2] * (s * b)
        nrm = torch.nn.functional.normalize(torch.linalg.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]), dim=1)
        lo, hi = tri.amin((0, 1)), tri.amax((0, 1))
        if rays == "shadow":  # towards points above the scene
            q = lo + (hi - lo) * (rnd(n, 3) * torch.tensor([1.0, 0.5, 1.0], device="cuda") +
                                  torch.tensor([0.0, 0.5, 0.0], device="cuda"))
            d = q - p
            length = d.norm(dim=1, keepdim=True).clamp_min(1e-6)
            d = d / length
            out[:, 7] = (length[:, 0] - 1e-3).clamp_min(0)
        else:
            d = torch.nn.functional.normalize(torch.randn(n, 3, generator=g, device="cuda"), dim=1) + nrm
            d = torch.nn.functional.normalize(d, dim=1)
        o = p + 1e-4 * nrm * (nrm * d).sum(1, keepdim=True).sign()
    out[:, 0:3], out[:, 4:7] = o, d
    return out


def prepare(case, seed):
    ctx = la.Context(0)
    scene = _scene(case, seed)
    s = dict(case=case, ctx=ctx, scene=scene)
    kind = case["kind"]
    if kind in ("trace", "rebuild"):
        s["rays"] = _rays(case, scene, seed)
        if kind == "trace":
            ctx.upload(scene)
            ctx.build_accel()
        n = case["n"]
        if case.get("any"):
            s["hits"] = torch.zeros(n, dtype=torch.uint8, device="cuda")
            s["out"] = {"occluded": s["hits"]}
        else:
            s["hits"] = torch.zeros(n, 5, dtype=torch.int32, device="cuda")  # lt_hit: t, prim, inst, u, v
            f = s["hits"].view(torch.float32)
            s["out"] = {"t": f[:, 0], "ids": s["hits"][:, 1:3], "uv": f[:, 3:5]}
    elif kind == "adjoint":
        s["adj"] = Adjoint(scene, ctx, case["width"], case["height"], spp=case["spp"], variants=case["variants"],
                           albedo_texture=0, roughness_texture=1, max_depth=case["depth"])
        base = [torch.from_numpy(np.ctypeslib.as_array(scene.desc.textures[t].data, shape=(
            scene.desc.textures[t].height, scene.desc.textures[t].width, 4)).copy()).cuda() for t in (0, 1)]
        g = torch.Generator("cuda").manual_seed(seed)
        vary = lambda shape: (torch.rand(shape, generator=g, device="cuda") - 0.5) * 0.4
        s["albedo"] = (base[0][None, ..., :3] + vary(s["adj"].albedo_shape)).clamp(0.05, 0.95).requires_grad_()
        s["rough"] = (base[1][None, ..., 0] + vary(s["adj"].rough_shape)).clamp(0.1, 0.95).requires_grad_()
        s["target"] = torch.rand(case["height"], case["width"], 3, generator=g, device="cuda")
        s["seed"] = seed & 0x7FFFFFFF
    else:
        kw = dict(width=case["width"], height=case["height"], path_length=case["depth"])
        if kind == "path":
            it = la.Path(scene, ctx, strategy=case["strategy"], **kw)
        elif kind == "bdpt":
            it = la.BDPT(scene, ctx, mis=case["mis"], **kw)
        elif kind == "vcm":
            it = la.VCM(scene, ctx, radius_factor=case["radius"], alpha=case["alpha"], enable_vm=case["vm"],
                        estimator=case["estimator"], **kw)
        else:
            it = la.SPPM(scene, ctx, base_radius=case["radius"], **kw)
        it.init()
        it.create_accel()
        it.seed = seed & 0x7FFFFFFF
        s["it"] = it
    ctx.synchronize()
    torch.cuda.synchronize()
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "rebuild":
        ctx.upload(s["scene"])
        ctx.build_accel()
    if kind in ("trace", "rebuild"):
        query = ctx.trace_any_device if case.get("any") else ctx.trace_closest_device
        query(s["rays"].data_ptr(), case["n"], s["hits"].data_ptr())
        return s["out"]
    if kind == "adjoint":
        img = render_textures(s["adj"], s["albedo"], s["rough"], s["seed"], case["cache"])
        loss = ((img - s["target"]) ** 2).sum()
        ga, gr = torch.autograd.grad(loss, (s["albedo"], s["rough"]))
        return {"image": img.detach(), "grad_albedo": ga, "grad_rough": gr}
    it = s["it"]
    it.reset()
    it.render(spp=case["spp"])
    return it.output_tex


# ------------------------------------------------------- work, tolerances ----
def work(case):
    """Scene, inputs and outputs once; per query one root-to-leaf descent of an
    8-wide tree (8 box tests of 18 operations a level) and one triangle test."""
    kind, tris = case["kind"], case["tris"]
    per_ray = 144.0 * max(1.0, math.log(max(tris, 8), 8)) + 60.0
    scene = tris * 48.0
    if kind in ("trace", "rebuild"):
        out = 1.0 if case.get("any") else 20.0
        return {"bytes": scene * (3.0 if kind == "rebuild" else 1.0) + case["n"] * (32.0 + out),
                "flops": case["n"] * per_ray + (tris * 200.0 if kind == "rebuild" else 0.0)}
    px = float(case["width"] * case["height"])
    if kind == "adjoint":
        samples = px * case["variants"] * case["spp"]
        texels = case["variants"] * case["tex"] ** 2 * 16.0
        return {"bytes": scene + 2 * texels + 2 * 12.0 * px * case["variants"],
                "flops": samples * 2.0 * (2 * per_ray + 300.0)}
    # rays per pixel and frame that every estimator of the kind casts: a camera
    # ray and its light ray; the bidirectional ones as many again from the light
    rays = 2.0 if kind == "path" else 4.0
    return {"bytes": scene + 16.0 * px, "flops": px * case["spp"] * rays * (per_ray + 150.0)}


# Hits are exact (watertight test, ties to the smaller triangle).  Images hold
# paths whose discrete choices flip on a last-bit difference: the same kernels
# without fused multiply-adds differ from these by rel 2.9e-4, max 0.25 (path,
# terrain), 8.5e-5, 0.012 (bdpt), 1e-5, 0.0016 (vcm), 1.5e-4, 0.15 (sppm),
# 2e-5, 0.014 (adjoint); about four times that, and room for one flipped path
# in a small image.
_TOL = {"path": (2e-3, 0.99), "bdpt": (1e-3, 0.5), "vcm": (5e-4, 0.5), "sppm": (1e-3, 0.9), "adjoint": (2e-4, 0.1)}


def tolerance(case):
    if case["kind"] not in _TOL:
        return "exact"
    rel, most = _TOL[case["kind"]]
    return {"rel": rel, "max": most}


# ------------------------------------------------------- 64-bit references ----
def _brute(tri, o, d, tmin, tmax):
    """(t, index, u, v) of the nearest triangle per ray in float64 (index -1: none)."""
    n = len(o)
    best = torch.full((n,), math.inf, dtype=torch.float64, device=o.device)
    idx = torch.full((n,), -1, dtype=torch.int64, device=o.device)
    bu, bv = torch.zeros_like(best), torch.zeros_like(best)
    e1, e2, v0 = tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0], tri[:, 0]
    step = max(1, int(3e7 // max(n, 1)))
    for a in range(0, len(tri), step):
        E1, E2, V0 = e1[a:a + step], e2[a:a + step], v0[a:a + step]
        p = torch.linalg.cross(d[:, None], E2[None])
        det = (E1 * p).sum(-1)
        s = o[:, None] - V0
        u = (s * p).sum(-1) / det
        q = torch.linalg.cross(s, E1[None].expand_as(s))
        v = (d[:, None] * q).sum(-1) / det
        t = (E2 * q).sum(-1) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= tmin[:, None]) & (t <= tmax[:, None])
        t = torch.where(ok, t, math.inf)
        m, j = t.min(1)
        better = m < best
        best = torch.where(better, m, best)
        idx = torch.where(better, j + a, idx)
        bu = torch.where(better, u.gather(1, j[:, None])[:, 0], bu)
        bv = torch.where(better, v.gather(1, j[:, None])[:, 0], bv)
    return best, idx, bu, bv


def _exact_hits(case, seed):
    if case.get("any") or case["n"] * float(case["tris"]) > 2e10:
        return None  # occlusion bits have no rounding; larger products take minutes
    scene = _scene(case, seed)
    r = _rays(case, scene, seed).double()
    tri = torch.from_numpy(scene.triangles()).cuda().double()
    t, u, v = (torch.zeros(case["n"], dtype=torch.float64, device="cuda") for _ in range(3))
    for a in range(0, len(r), 65536):
        q = r[a:a + 65536]
        bt, bi, uu, vv = _brute(tri, q[:, 0:3], q[:, 4:7], q[:, 3], q[:, 7])
        hit = bi >= 0
        t[a:a + 65536], u[a:a + 65536], v[a:a + 65536] = torch.where(hit, bt, 0.0), torch.where(hit, uu, 0.0), \
            torch.where(hit, vv, 0.0)
    return {"t": t, "ids": None, "uv": torch.stack([u, v], 1)}


class _Pcg:
    """pcg4d streams of (x, y, frame, counter), one per lane (uniform floats of 23 bits)."""

    def __init__(self, x, y, frame):
        self.x, self.y, self.z, self.w = x, y, torch.full_like(x, frame), torch.zeros_like(x)

    def __call__(self, live):
        M = 0xFFFFFFFF
        self.w = self.w + live.long()
        x, y, z, w = ((c * 1664525 + 1013904223) & M for c in (self.x, self.y, self.z, self.w))
        x = (x + y * w) & M
        y = (y + z * x) & M
        z = (z + x * y) & M
        w = (w + y * z) & M
        x, y, w = x ^ (x >> 16), y ^ (y >> 16), w ^ (w >> 16)
        return (((x + y * w) & M) >> 9).double() / (1 << 23)


def _exact_path(case, seed):
    """The Path estimator on the Cornell box (Lambert surfaces, one area light)
    in float64: NEE with MIS, roulette after depth 3, its stale-hit rule for
    MIS rays that leave the box."""
    W, H, dev, f64 = case["width"], case["height"], "cuda", torch.float64
    if case["scene"] != "cornell" or W * H * case["spp"] * case["depth"] > 3e7:
        return None  # more triangles, or more samples, take minutes by brute force
    scene = _scene(case, seed)
    d = scene.desc
    tri = torch.from_numpy(scene.triangles()).to(dev, f64)
    counts = scene._mesh_ranges()[1] // 3
    mesh = torch.from_numpy(np.repeat(np.arange(d.num_prim_infos), counts)).to(dev)
    first = np.concatenate([[0], np.cumsum(counts)])
    vert = np.ctypeslib.as_array(C.cast(d.vertices, C.POINTER(C.c_float)), shape=(d.num_vertices, 8))
    idx = np.ctypeslib.as_array(d.indices, shape=(d.num_indices,)).astype(np.int64)
    vo = np.repeat([d.prim_infos[m].vertex_offset for m in range(d.num_prim_infos)], counts)
    nrm = torch.from_numpy(vert[idx.reshape(-1, 3) + vo[:, None], 3:6].copy()).to(dev, f64)
    mats = [d.materials[d.prim_infos[m].material_index] for m in range(d.num_prim_infos)]
    alb = torch.tensor([list(m.albedo) for m in mats], dtype=f64, device=dev)
    emi = torch.tensor([list(m.emissive_factor) for m in mats], dtype=f64, device=dev)
    light, n_light = int(d.lights[0].prim_mesh_idx), int(d.lights[0].num_triangles)
    unit = lambda a: a / a.norm(dim=1, keepdim=True)
    dot = lambda a, b: (a * b).sum(1)
    sky = torch.tensor(list(scene.integrator_cfg().sky_col), dtype=f64, device=dev)
    cam = scene.camera(W, H)
    inv_v = torch.tensor(list(cam.inv_view), dtype=f64, device=dev).view(4, 4).T
    inv_p = torch.tensor(list(cam.inv_projection), dtype=f64, device=dev).view(4, 4).T

    def closest(o, dd):
        lim = torch.ones(len(o), dtype=f64, device=dev)
        t, i, u, v = _brute(tri, o, dd, lim * 0.001, lim * 1e4)
        hit, i = i >= 0, i.clamp_min(0)
        b = torch.stack([1 - u - v, u, v], 1)[..., None]
        ng = unit(torch.linalg.cross(tri[i, 2] - tri[i, 0], tri[i, 1] - tri[i, 0]))
        return hit, i, (tri[i] * b).sum(1), unit((nrm[i] * b).sum(1)), ng

    def hemisphere(n, r0, r1):
        ox, oy = 2 * r0 - 1, 2 * r1 - 1
        wide = ox.abs() > oy.abs()
        r = torch.where(wide, ox, oy)
        th = torch.where(wide, 0.25 * math.pi * oy / torch.where(ox == 0, 1.0, ox),
                         math.pi * (0.5 - 0.25 * ox / torch.where(oy == 0, 1.0, oy)))
        x, y = r * th.cos(), r * th.sin()
        z = (1 - x * x - y * y).clamp_min(0).sqrt()
        sg = torch.where(n[:, 2] >= 0, 1.0, -1.0)
        a = -1 / (sg + n[:, 2])
        b = n[:, 0] * n[:, 1] * a
        t1 = torch.stack([1 + sg * n[:, 0] ** 2 * a, sg * b, -sg * n[:, 0]], 1)
        t2 = torch.stack([b, sg + n[:, 1] ** 2 * a, -n[:, 1]], 1)
        return x[:, None] * t1 + y[:, None] * t2 + z[:, None] * n, z

    def offset(p, n):  # a few units in the last place of the 32-bit position
        f = p.float()
        k = (256 * n).trunc().int()
        near = (f.view(torch.int32) + torch.where(f < 0, -k, k)).view(torch.float32).double() - f.double() + p
        return torch.where(p.abs() < 1 / 32, p + n / 65536, near)

    pix = torch.arange(W * H, device=dev)
    total = torch.zeros(W * H, 3, dtype=f64, device=dev)
    for frame in range(case["spp"]):
        rng = _Pcg(pix % W, pix // W, frame ^ (seed & 0x7FFFFFFF))
        live = torch.ones(W * H, dtype=torch.bool, device=dev)
        ux, uy = ((c.double() + rng(live)) / s for c, s in ((pix % W, W), (pix // W, H)))
        ndc = torch.stack([2 * ux - 1, 2 * uy - 1, torch.ones_like(ux), torch.ones_like(ux)], 1)
        o, dd = inv_v[:3, 3].expand(W * H, 3), unit((ndc @ inv_p.T)[:, :3]) @ inv_v[:3, :3].T
        col, thr = torch.zeros_like(total), torch.ones_like(total)
        for depth in range(case["depth"]):
            hit, i, p, ns, ng = closest(o, dd)
            col += torch.where((live & ~hit)[:, None], thr * sky, 0.0)
            live = live & hit
            m = mesh[i]
            if depth == 0:
                col += torch.where(live[:, None], thr * emi[m], 0.0)
            if depth >= case["depth"] - 1:
                break
            wo = -dd
            ng = torch.where((dot(ng, wo) < 0)[:, None], -ng, ng)
            ns = torch.where((dot(ng, ns) < 0)[:, None], -ns, ns)
            f = alb[m] / math.pi
            rng(live)
            lt = (rng(live) * n_light).long()
            r2, r3 = rng(live).sqrt(), rng(live)
            gl = int(first[light]) + lt
            bc = torch.stack([r2 - r3 * r2, 1 - r2, r3 * r2], 1)[..., None]
            q, qn = (tri[gl] * bc).sum(1), unit((nrm[gl] * bc).sum(1))
            pdf_a = 2 / torch.linalg.cross(tri[gl, 1] - tri[gl, 0], tri[gl, 2] - tri[gl, 0]).norm(dim=1)
            wi = q - p
            dist = wi.norm(dim=1)
            wi = wi / dist[:, None]
            Le, start = emi[light], p + (2 / 65536) * ns
            cx, pdf_w = dot(ns, wi), pdf_a * dist ** 2 / dot(qn, -wi).abs()
            zo = dot(ns, wo)
            ok = torch.minimum(cx, zo) > 0
            c = torch.where(ok, cx.abs() / (1 + cx / math.pi / pdf_w) / pdf_w, 0.0)
            zero = torch.zeros_like(dist)
            seen = _brute(tri, start, wi, zero, dist - 0.001)[1] < 0
            res = torch.where((seen & live)[:, None], c[:, None] * f * Le, 0.0)
            s0, s1 = rng(live), rng(live)
            rng(live)
            wb, z = hemisphere(ns, s0, s1)
            h2, i2, p2, n2, _ = closest(start, wb)
            n2, p2, i2 = torch.where(h2[:, None], n2, ns), torch.where(h2[:, None], p2, p), torch.where(h2, i2, i)
            g = dot(n2, -wb).abs() / (p2 - p).norm(dim=1) ** 2
            w = torch.where((z > 0) & (zo > 0), math.pi / (1 + pdf_a / (g * z / math.pi)), 0.0)
            res += torch.where(((i2 == gl) & live & (z > 0))[:, None], w[:, None] * f * Le, 0.0)
            col += thr * res * n_light
            s0, s1 = rng(live), rng(live)
            rng(live)
            o = offset(p, ng)
            dd, z = hemisphere(ns, s0, s1)
            live = live & (z > 0)
            thr = thr * torch.where(((zo > 0) & (z > 0))[:, None], f * math.pi, 0.0)
            if depth > 3:
                pr = (thr @ torch.tensor([0.2126, 0.7152, 0.0722], dtype=f64, device=dev)).clamp_max(0.95)
                live = live & (pr != 0) & (pr >= rng(live))
                thr = thr / torch.where(live, pr, 1.0)[:, None]
        total += col
    out = torch.ones(H, W, 4, dtype=f64, device=dev)
    out[..., :3] = (total / case["spp"]).view(H, W, 3)
    return out.cpu().numpy()


def exact(case, seed):
    if case["kind"] in ("trace", "rebuild"):
        return _exact_hits(case, seed)
    if case["kind"] == "path":
        return _exact_path(case, seed)
    return None  # whole bidirectional and textured estimators over meshes: minutes by brute force
