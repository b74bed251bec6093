"""The adjoint interleaves the variants' texels and shares a sample's rays
between its variants where these pay (csrc/adjoint.h).  Each variant must come
out bit for bit as if rendered alone (one variant: neither is done), whatever
the variants, the samples and the depth: variants that fill no, one or several
waves, more samples than one shared walk holds, more bounces than are kept,
and texels that send nearly every path its own way.  path_blocks_per_cu = 1
makes the grid small, so that the small images here have the groups per wave
from which on rays are shared."""
import numpy as np
import pytest

import lumen_amd as la
from test_gpu_adjoint import _cmp_grad, _scene, _variants

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("W,H,V,spp,depth,swap", [
    # not shared: too few variants, groups per wave, lanes
    (24, 16, 4, 3, 6, False),
    (8, 8, 64, 4, 5, True),
    (160, 128, 16, 1, 3, False),
    # shared: runs of 4 and 2 groups, variants that straddle waves and edge tiles cut
    (256, 128, 32, 8, 5, True),
    (160, 150, 23, 8, 6, False),
    (150, 131, 23, 12, 6, True),
    # more samples than a shared walk holds; a pixel over several waves
    (64, 60, 100, 70, 3, True),
    # bounces beyond the kept ones, camera rays only
    (128, 128, 16, 16, 20, False),
    (128, 128, 16, 16, 1, False),
])
def test_variants_match_single_renders(gpu_ctx, W, H, V, spp, depth, swap):
    print(f"[gpu] adjoint shared rays {W}x{H} V={V} spp={spp} depth={depth}", flush=True)
    from lumen_amd.adjoint import Adjoint
    sc, alb, rough = _scene()
    rng = np.random.default_rng(V + depth)
    albs, roughs = _variants(alb, rough, V, rng)
    if swap:  # black texels in the first variant (its walk ends early) and unlike roughness
        albs[0, ::2] = 0.0
        roughs[1::2] = 1.0 - 0.9 * roughs[1::2]
    ta, tr = torch.from_numpy(albs).cuda(), torch.from_numpy(roughs).cuda()
    w = torch.from_numpy(rng.normal(size=(V, H, W, 3)).astype(np.float32)).cuda()
    gpu_ctx.set_tuning(path_blocks_per_cu=1)
    kw = dict(spp=spp, albedo_texture=0, roughness_texture=1, max_depth=depth)
    adj = Adjoint(sc, gpu_ctx, W, H, variants=V, **kw)
    one = Adjoint(sc, gpu_ctx, W, H, variants=1, **kw)
    gpu_ctx.set_tuning()
    img, cache = adj.forward(ta, tr, seed=11)
    again, _ = adj.forward(ta, tr, seed=11, cache=False)
    ga, gr = adj.backward(ta, tr, w, seed=11, cache=cache)
    adj.set_counting(True)
    img_c, _ = adj.forward(ta, tr, seed=11)
    cnt = adj.counts()
    torch.cuda.synchronize()
    assert torch.equal(img, again) and torch.equal(img, img_c)
    one.set_counting(True)
    rays = np.zeros(2, np.int64)
    for v in sorted({0, 1, V // 2, V - 1}):
        iv, cv = one.forward(ta[v:v + 1].contiguous(), tr[v:v + 1].contiguous(), seed=11)
        c = one.counts()
        rays += (c["closest"], c["shadow"])
        assert torch.equal(iv[0], img[v]), f"variant {v}"
        if v in (0, V - 1):
            a1, r1 = one.backward(ta[v:v + 1].contiguous(), tr[v:v + 1].contiguous(), w[v:v + 1], seed=11, cache=cv)
            _cmp_grad(ga[v].cpu().numpy(), a1[0].cpu().numpy(), f"albedo gradient v{v}")
            _cmp_grad(gr[v].cpu().numpy(), r1[0].cpu().numpy(), f"roughness gradient v{v}")
    # a ray is counted for each variant that takes it (all variants: V at most)
    assert W * H * spp * V <= cnt["closest"] and cnt["shadow"] >= rays[1]
    if V <= 4:
        assert (cnt["closest"], cnt["shadow"]) == tuple(rays)
    adj.close()
    one.close()
