"""The dense grid's walk: many cells found, then loaded together.

Grids from one voxel up and around multiples of the 16 cells that are found at
a time; eyes inside, outside, on whole coordinates, and so far away that the
general walk takes the ray; rays whose planes on two axes are crossed at one t
up to the grid's edge, where the last cell is entered at the t the ray leaves;
shadows and occlusion rays, which end at a distance.
"""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R

from test_gpu_variants import _check, _fresh

pytestmark = pytest.mark.gpu

LIGHT = (0.4, 1.0, 0.3)


def _compare(ctx, grid, views, flags, what):
    n = grid.shape[0]
    sc = ctx.scene_dense(grid)
    osc = O.dense_scene(grid.ravel())
    hits = 0
    for k, (eye, target, up, vfov, w, h) in enumerate(views):
        cam = R.camera(eye, target, up, vfov, w, h)
        ocam = O.camera(eye, target, up, vfov, w, h)
        sh = (LIGHT, 9, 4, 6.0)
        ref = O.raymarch(osc, ocam, flags, O.shading(*sh), threads=4)
        hits += int((ref[1] < 6).sum())
        tg = R.RayTargets(ctx, w, h, index_bytes=8, counters=True)
        for count in (0, L.RAY_COUNT):  # the general walk counts steps
            _fresh(tg)
            R.raymarch(ctx, sc, cam, flags | count, R.shading(*sh), tg)
            ctx.sync()
            _check(ctx, tg, ref, "%s n=%d view %d" % (what, n, k), count=bool(count))
    sc.destroy()
    return hits


@pytest.mark.parametrize("n", [1, 2, 3, 15, 16, 17, 31, 33, 65])
def test_grids_and_eyes(ctx, n):
    rng = np.random.default_rng(n)
    grid = (rng.random((n, n, n)) < (0.5 if n < 4 else 0.01)).astype(np.uint8)
    grid[n // 2, n // 2, n // 2] = 1
    m, up = n / 2.0, (0.0, 1.0, 0.0)
    far = 70000.0
    views = [
        ((-0.4 * n, 1.3 * n, 1.6 * n), (m, m, m), up, 50.0, 65, 43),
        ((float(2 * n), float(n), float(n)), (0.0, 0.0, 0.0), up, 40.0, 33, 31),
        ((m + 0.25, 0.3 * n, m), (n, 0.6 * n, 0.2 * n), up, 90.0, 40, 40),
        ((m, float(3 * n), m), (m, 0.0, m), (0.0, 0.0, 1.0), 30.0, 1, 17),
        ((far, far * 0.9, m), (m, m, m), up, 0.002 * n, 24, 24),
    ]
    flags = L.RAY_SHADOW | L.RAY_AO
    assert _compare(ctx, grid, views, flags, "eyes") > 0


@pytest.mark.parametrize("n", [5, 16, 40])
@pytest.mark.parametrize("sign", [1, -1])
def test_cell_entered_at_the_exit(ctx, n, sign):
    # one pixel column: d.x equals d.z in every ray, and the eye's x and z
    # differ by a whole number, so x and z planes are crossed together, x
    # first.  The wall is the cells a ray enters by x as it leaves by z.
    gap, y = 2, n / 2.0
    if sign > 0:
        eye, target, x, z = (-4.5, y, -4.5 + gap), (n - 4.5, y, n - 4.5 + gap), n - gap, n - 1
    else:
        eye = (n + 4.5, y, n + 4.5 - gap)
        target, x, z = (4.5, y, 4.5 - gap), gap - 1, 0
    grid = np.zeros((n, n, n), np.uint8)
    grid[z, :, x] = 7
    hits = _compare(ctx, grid, [(eye, target, (0.0, 1.0, 0.0), 50.0, 1, 65)], L.RAY_SHADOW, "exit")
    assert hits > 0
