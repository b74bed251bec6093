"""The merge pass's split of heavy queries and its photon buckets: a merge
radius so large that every query holds many parts of photons, images of one
tile and of ragged tiles (the query segments), radii from a sliver to the
whole scene (runs of cells across bucket runs, negative cells), against the
oracle."""
import numpy as np
import pytest

import lumen_amd as la
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,size,radius,depth", [
    ("cornell", (8, 8), 60.0, 4),      # a few hundred photons, one tile
    ("cornell", (75, 50), 80.0, 5),    # ~10,000 photons a query: several parts each
    ("cornell", (75, 50), 3.0, 5),
    ("caustics", (90, 61), 6.0, 6),    # a few heavy queries among light ones
    ("caustics", (65, 9), 0.05, 6),
])
def test_merges_match_the_oracle(gpu_ctx, kind, size, radius, depth):
    print(f"[gpu] vcm merges {kind} {size} radius {radius}", flush=True)
    W, H = size
    sc = la.Scene.procedural(kind, seed=2, **({"sphere_tris": 2000} if kind == "caustics" else {}))
    it = la.VCM(sc, gpu_ctx, W, H, path_length=depth, radius_factor=radius, alpha=0.75, enable_vm=True,
                estimator="corrected")
    it.init()
    it.create_accel()
    it.set_counting(True)
    it.render(spp=2)
    img, st = it.output_tex, it.stats()
    acc = oracle.Accel(sc.desc)
    ref = acc.render_vcm(it.camera, W, H, depth, frames=2, radius_factor=radius, alpha=0.75, use_vm=True,
                         corrected=True)[0]
    a, b = img[..., :3], ref[..., :3]
    # the replay bar of the VCM tests: sums reordered by the atomics, rare
    # flips of a discrete choice by a last-bit difference
    ok = np.all(np.abs(a - b) <= 1e-3 * (1 + np.abs(b)), axis=-1).mean()
    rel = np.sqrt(((a - b) ** 2).sum() / (b ** 2).sum())
    print(f"[gpu] {ok:.4f} of the pixels, rel {rel:.2e}, photons gathered {st.photons_gathered}", flush=True)
    assert ok >= 0.995 and rel <= 0.01
    assert st.photons_gathered > 0 or radius < 0.1
    it.destroy()
