"""The VCM photon grids of scenes that are thin or flat along an axis
(lumen_amd/csrc/vcm_grid.h): the cells a merge query visits stay few, and every
photon within the radius lies in one of them.  The arithmetic is compiled for
the host; a GPU would run a range of 2^29 cells for minutes."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

import lumen_amd as la
import oracle
from scenes import DescScene, camera

ROOT = Path(__file__).resolve().parents[1]
SRC = r"""
#include "vcm_grid.h"
extern "C" void query(const float* lo, const float* hi, float radius, const int* res, const float* q, const float* p,
                      int n, int* runs, int* outside) {
    float inv[3];
    for (int k = 0; k < 3; k++) inv[k] = vcm_inv_ext(lo[k], hi[k], radius, res[k]);
    int a[3], b[3];
    for (int k = 0; k < 3; k++) {
        a[k] = vcm_cell(q[k] - radius, lo[k], inv[k], res[k]);
        b[k] = vcm_cell(q[k] + radius, lo[k], inv[k], res[k]);
    }
    *runs = vcm_runs(a, b).n;
    *outside = 0;
    for (int i = 0; i < n; i++)
        for (int k = 0; k < 3; k++) {
            const int c = vcm_cell(p[3 * i + k], lo[k], inv[k], res[k]);
            if (c < a[k] || c > b[k]) ++*outside;
        }
}
extern "C" float reference_bmax(float lo, float hi, float radius, int res) { return vcm_reference_bmax(lo, hi, radius, res); }
"""


@pytest.fixture(scope="module")
def grid(tmp_path_factory):
    d = tmp_path_factory.mktemp("vcm_grid")
    (d / "g.cpp").write_text(SRC)
    subprocess.run([shutil.which("g++") or "g++", "-O1", "-std=c++17", "-shared", "-fPIC",
                    f"-I{ROOT / 'lumen_amd' / 'csrc'}", str(d / "g.cpp"), "-o", str(d / "g.so")], check=True)
    L = C.CDLL(str(d / "g.so"))
    L.reference_bmax.restype = C.c_float
    L.reference_bmax.argtypes = [C.c_float, C.c_float, C.c_float, C.c_int]
    return L


def _bounds(axis, ext, at=0.25):
    lo, hi = np.float32([-1, -2, -1.5]), np.float32([1, 2, 1.5])
    lo[axis] = at
    hi[axis] = np.float32(at) + np.float32(ext)
    return lo, hi


def _res(lo, hi, radius, div):
    base = int((hi - lo).max() / radius)
    return np.maximum(((hi - lo) * base / (hi - lo).max()).astype(np.int32), 1) * div


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("ext,at", [(0.0, 0.25), (0.0, 0.0), (1e-40, 0.0), (1e-30, 0.0), (1e-6, 0.25), (1e-6, 0.0),
                                    (0.004, 0.25), (0.006, 0.25), (0.013, 0.25), (1.0, 0.25)])
def test_query_range_is_bounded_and_complete(grid, axis, ext, at):
    radius = np.float32(0.01)
    lo, hi = _bounds(axis, ext, at)
    res = np.ascontiguousarray(_res(lo, hi, radius, 2), np.int32)
    rng = np.random.default_rng(3)
    worst = 0
    for _ in range(200):
        q = rng.uniform(lo, hi).astype(np.float32)
        d = rng.normal(size=(64, 3))
        d *= (float(radius) * rng.random((64, 1)) / np.linalg.norm(d, axis=1, keepdims=True))
        p = np.ascontiguousarray((q + d).astype(np.float32))
        p[:, axis] = np.clip(p[:, axis], lo[axis], hi[axis])
        n, out = C.c_int(), C.c_int()
        P = lambda a: a.ctypes.data_as(C.c_void_p)
        grid.query(P(lo), P(hi), C.c_float(radius), P(res), P(q), P(p), len(p), C.byref(n), C.byref(out))
        assert out.value == 0
        worst = max(worst, n.value)
    # at most 4 * 2 + 1 cells of x and y, which along z touch at most 2 + 1 runs of 8
    assert 1 <= worst <= 9 * 9 * 3


def test_reference_grid_keeps_its_bounds_unless_flat(grid):
    assert grid.reference_bmax(0.25, 0.25, 0.01, 1) == np.inf
    assert grid.reference_bmax(0.0, 1e-30, 0.01, 1) == np.inf
    for lo, hi, res in [(0, 1e-6, 1), (-1, 1, 200), (0, 0.005, 1), (1, -1, 1)]:
        assert grid.reference_bmax(lo, hi, 0.01, res) == np.float32(hi)


class _FlatWall:
    """A quad at z = 0 lit by a point light, whose own bounds have no extent in z."""

    def __init__(self):
        s = DescScene()
        m = s.material(bsdf_type=1, bsdf_props=9, albedo=(0.7, 0.6, 0.5))
        s.mesh([[[-1, -1, 0], [1, -1, 0], [1, 1, 0]], [[-1, -1, 0], [1, 1, 0], [-1, 1, 0]]], m)
        s.analytic.append(dict(pos=(0.3, 0.2, 0.8), to=(0, 0, 0), L=(4, 4, 4), flags=4 | 16 | 32))
        self.s, self.desc, self._h = s, s.build(), None

    def camera(self, w, h):
        return camera([0, 0, 2.5], [0, 0, -1], 45, w / h)

    def integrator_cfg(self):
        return la._abi.lt_scene_integrator_cfg()


@pytest.mark.gpu
@pytest.mark.parametrize("estimator", ["corrected", "reference"])
def test_flat_wall_merges(gpu_ctx, estimator):
    print(f"[gpu] vcm flat wall {estimator}", flush=True)
    W, H, depth, radius = 48, 40, 4, 4.0
    sc = _FlatWall()
    assert sc.desc.scene_min[2] == sc.desc.scene_max[2]
    it = la.VCM(sc, gpu_ctx, W, H, path_length=depth, sky_col=(0, 0, 0), radius_factor=radius, alpha=0.75,
                enable_vm=True, estimator=estimator)
    it.init()
    it.create_accel()
    it.set_counting(True)
    it.render(spp=2)
    img, st = it.output_tex[..., :3], it.stats()
    it.destroy()
    acc = oracle.Accel(sc.desc)
    ref = acc.render_vcm(it.camera, W, H, depth, frames=2, radius_factor=radius, alpha=0.75, use_vm=True,
                         corrected=estimator == "corrected")[0][..., :3]
    # the replay bar of the VCM tests
    ok = np.all(np.abs(img - ref) <= 1e-3 * (1 + np.abs(ref)), axis=-1).mean()
    rel = np.sqrt(((img - ref) ** 2).sum() / (ref ** 2).sum())
    print(f"[gpu] {ok:.4f} of the pixels, rel {rel:.2e}, photons gathered {st.photons_gathered}", flush=True)
    assert ref.sum() > 0 and ok >= 0.995 and rel <= 0.01
    assert estimator == "reference" or st.photons_gathered > 0
