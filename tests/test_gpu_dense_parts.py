"""Small dense frames, whose rays four lanes walk, against the oracle: the
default launch and 16x16 tiles (a lane per pixel), grids around the walk's
batches, eyes inside, outside, on whole coordinates and far away, rays along
an axis and through a grid's corners, and frame sizes on both sides of the
line between the two kernels (256 CUs)."""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R

from test_gpu_variants import _check, _force, _fresh

pytestmark = pytest.mark.gpu

UP = (0.0, 1.0, 0.0)


def _both(ctx, tmp_path, grid, view, light, radius):
    n, (w, h) = grid.shape[0], view[4:]
    flags = L.RAY_SHADOW | L.RAY_AO
    sc, osc = ctx.scene_dense(grid), O.dense_scene(grid.ravel())
    sh = (light, 5, 5, radius)  # five samples over four lanes
    ref = O.raymarch(osc, O.camera(*view), flags, O.shading(*sh), threads=4)
    tg = R.RayTargets(ctx, w, h)
    for shape in [None, (0, 16, 16, 0), (2, 8, 8, 0)]:
        if shape:
            _force(ctx, tmp_path, L.SCENE_DENSE_U8, n, w, h, flags, shape)
        _fresh(tg)
        R.raymarch(ctx, sc, R.camera(*view), flags, R.shading(*sh), tg)
        ctx.sync()
        _check(ctx, tg, ref, "n=%d %s %s" % (n, view, shape), count=False)
    sc.destroy()
    return int((ref[1] < 6).sum())


@pytest.mark.parametrize("n", [1, 2, 16, 35, 64])
@pytest.mark.parametrize("light", [(0.4, 1.0, 0.3), (0.0, 1.0, 0.0)])
def test_grids_and_eyes(ctx, tmp_path, n, light):
    rng = np.random.default_rng(n)
    grid = (rng.random((n, n, n)) < (0.5 if n < 4 else 0.006)).astype(np.uint8)
    grid[n // 2, n // 2, n // 2] = 1
    m = n / 2.0
    views = [
        ((-0.4 * n, 1.3 * n, 1.6 * n), (m, m, m), UP, 50.0, 47, 31),
        ((float(2 * n), float(2 * n), float(2 * n)), (0.0, 0.0, 0.0), UP, 40.0, 35, 33),
        ((m + 0.25, 0.3 * n, m), (n, 0.6 * n, 0.2 * n), UP, 90.0, 38, 38),
        ((m, float(3 * n), m), (m, 0.0, m), (0.0, 0.0, 1.0), 30.0, 1, 19),
        ((-3.0, 0.5, 0.5), (n, 0.5, 0.5), UP, 20.0, 21, 1),
        ((70000.0, 63000.0, m), (m, m, m), UP, 0.002 * n, 26, 22),
    ]
    assert sum(_both(ctx, tmp_path, grid, v, light, 7.0) for v in views) > 0


@pytest.mark.parametrize("n", [7, 33])
@pytest.mark.parametrize("sign", [1, -1])
def test_cell_entered_at_the_exit(ctx, tmp_path, n, sign):
    # planes of x and z crossed together, x first; the wall is entered by x at
    # the t the ray leaves by z
    gap, y = 2, n / 2.0
    if sign > 0:
        eye, target, x, z = (-4.5, y, -4.5 + gap), (n - 4.5, y, n - 4.5 + gap), n - gap, n - 1
    else:
        eye, target, x, z = (n + 4.5, y, n + 4.5 - gap), (4.5, y, 4.5 - gap), gap - 1, 0
    grid = np.zeros((n, n, n), np.uint8)
    grid[z, :, x] = 7
    assert _both(ctx, tmp_path, grid, (eye, target, UP, 50.0, 1, 65), (0.4, 1.0, 0.3), 5.0) > 0


# 16384 tiles of 4x4 pixels, and a column more
@pytest.mark.parametrize("size", [(512, 512), (513, 512), (4, 16384), (1, 1), (3, 5)])
def test_frame_sizes(ctx, tmp_path, size):
    grid = O.spheres_dense(3, 24, 3)
    view = ((37.0, 30.0, 33.0), (11.0, 12.0, 13.0), UP, 55.0) + size
    _both(ctx, tmp_path, np.asarray(grid, np.uint8), view, (0.4, 1.0, 0.3), 4.0)
