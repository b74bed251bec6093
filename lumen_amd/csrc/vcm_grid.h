// vcm_grid.h — the VCM photon grids along one axis and the cells that a merge
// query visits (VCM.cpp:140-158, vcm_commons.glsl:19-23, 251-262).  Plain C++,
// so that the bounds below can be checked on the host.
#pragma once
#include <math.h>
#include <stdint.h>

#if defined(__HIP__) || defined(__HIPCC__)
#define LT_VCM_HD __host__ __device__ __forceinline__
#else
#define LT_VCM_HD inline
#endif

// The corrected estimator's cells are this many times finer per axis than the
// reference's: about radius / LT_VCM_CELL_DIV wide.
#ifndef LT_VCM_CELL_DIV
#define LT_VCM_CELL_DIV 2
#endif
// its cells follow one another along z in runs of 2^kRunBits (vcm.hip)
constexpr int kRunBits = 3;

// 1 / (bmax - bmin) of an axis of the corrected estimator's grid of `res`
// cells, but no finer than the merge radius asks for: an axis thinner than half
// the radius (a flat scene: no extent at all) gets cells of radius /
// LT_VCM_CELL_DIV, so that a query covers at most 4 LT_VCM_CELL_DIV + 1 cells
// of any axis.  Its sums do not depend on the grid.
LT_VCM_HD float vcm_inv_ext(float bmin, float bmax, float radius, int res) {
    const float inv = 1.0f / (bmax - bmin);
    if (inv > 0.0f && radius * inv * (float)res <= 2.0f * (float)LT_VCM_CELL_DIV) return inv;
    return (float)LT_VCM_CELL_DIV / (radius * (float)res);
}
LT_VCM_HD int vcm_cell(float p, float bmin, float inv_ext, int res) {
    return (int)((p - bmin) * inv_ext * (float)res);
}

// The reference estimator's upper bound of an axis: where a query would visit
// more than 2^20 cells along it (a flat scene: without end) every position is
// in cell 0.
LT_VCM_HD float vcm_reference_bmax(float bmin, float bmax, float radius, int res) {
    const float ext = bmax - bmin;
    return ext >= 0.0f && !(2.0f * radius / ext * (float)res <= 1048576.0f) ? INFINITY : bmax;
}

// a query's columns of cells along z, each in `nr` runs from r0 on: `n` runs in all
struct VcmRuns {
    int r0, nr, ny, n;
};
LT_VCM_HD VcmRuns vcm_runs(const int lo[3], const int hi[3]) {
    VcmRuns r;
    r.r0 = lo[2] >> kRunBits;
    r.nr = (hi[2] >> kRunBits) - r.r0 + 1;
    r.ny = hi[1] - lo[1] + 1;
    r.n = (hi[0] - lo[0] + 1) * r.ny * r.nr;
    return r;
}
