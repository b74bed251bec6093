"""How a persistent grid shares its items (csrc/dev_work.h): ray batches and
images around one tile, one tile per wave and the tiles that come from the
counter, on grids of different sizes; and the frames of one launch against
frames launched one by one (bit-identical: a sample's arithmetic does not
depend on where it runs, and the running mean is folded in frame order)."""
import numpy as np
import pytest

import lumen_amd as la
import oracle
from raygen import random_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks", [1, 3, 8])
def test_ray_batches_around_the_tile_counts(gpu_ctx, blocks):
    """With b workgroups per CU a grid has 2 b CUs waves: batches of one ray
    to several rounds of tiles per wave, ragged ends included."""
    print(f"[gpu] ray batches, {blocks} workgroups per CU", flush=True)
    sc = la.Scene.procedural("cornell", seed=1)
    gpu_ctx.upload(sc)
    gpu_ctx.build_accel()
    cus, _ = gpu_ctx.device_info()
    before = gpu_ctx.get_tuning()
    gpu_ctx.set_tuning(trace_blocks_per_cu=blocks)
    try:
        per_round = 64 * 2 * blocks * cus
        tris = sc.triangles()
        acc = oracle.Accel(sc.desc)
        sizes = {1, 63, 65, 1023, per_round - 1, per_round, per_round + 1, 2 * per_round + 77, 5 * per_round - 63}
        rays = random_rays(tris, max(sizes), 3)
        ref, occ = acc.closest(rays), acc.any(rays)
        for n in sorted(sizes):
            g = gpu_ctx.trace_closest(rays[:n])
            assert np.array_equal(g.view(np.uint8), ref[:n].view(np.uint8)), n
            assert np.array_equal(gpu_ctx.trace_any(rays[:n]), occ[:n]), n
    finally:
        gpu_ctx.set_tuning(**before)


@pytest.mark.parametrize("strategy", ["persistent", "megakernel"])
@pytest.mark.parametrize("size", [(1, 1), (9, 7), (65, 33), (509, 383)])
def test_frames_of_one_launch_equal_single_frames(gpu_ctx, strategy, size):
    print(f"[gpu] multi-frame launch {strategy} {size}", flush=True)
    sc = la.Scene.procedural("cornell", seed=1)
    imgs = []
    for groups in ([1] * 7, [3, 4], [7]):
        it = la.Path(sc, gpu_ctx, size[0], size[1], strategy=strategy)
        it.seed = 11
        it.init()
        it.create_accel()
        for n in groups:
            it.render(spp=n)
            it.update()
        imgs.append(it.output_tex)
        it.destroy()
    assert np.array_equal(imgs[0], imgs[1]) and np.array_equal(imgs[0], imgs[2])
    assert np.isfinite(imgs[0]).all() and (imgs[0][..., 3] == 1).all()


@pytest.mark.parametrize("size", [(1, 1), (17, 15), (16, 16), (257, 1), (509, 383)])
def test_wavefront_queues_around_a_workgroup(gpu_ctx, size):
    """Queues of one item to many workgroups' worth: the wavefront form equals
    the persistent one up to float summation order (test_gpu_path.py's bound),
    and repeats itself bit for bit (a path's terms do not depend on its
    queue slot)."""
    print(f"[gpu] wavefront queues {size}", flush=True)
    sc = la.Scene.procedural("cornell", seed=1)
    imgs = []
    for strategy in ("wavefront", "wavefront", "persistent"):
        it = la.Path(sc, gpu_ctx, size[0], size[1], strategy=strategy)
        it.seed = 5
        it.init()
        it.create_accel()
        it.render(spp=3)
        it.update()
        imgs.append(it.output_tex)
        it.destroy()
    assert np.array_equal(imgs[0], imgs[1])
    np.testing.assert_allclose(imgs[0], imgs[2], rtol=1e-4, atol=1e-5)
