"""The brick scenes' walk against the oracle, with and without step counts.

Solid boxes that end inside a 32^3 and a 128^3 block, edges that are no
multiple of either, eyes inside, outside, on whole coordinates and far away,
rays along an axis (primary, shadow), and rays whose planes on two axes are
crossed at one t up to the box's end, where the last cell is entered at the t
the ray leaves.
"""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R

from test_gpu_variants import _check, _fresh

pytestmark = pytest.mark.gpu

UP = (0.0, 1.0, 0.0)


def _scenes(ctx, grid, two_level):
    n = grid.shape[0]
    slots, masks, vox = O.brickmap_from_dense(grid)
    if not two_level:
        return ctx.scene_brickmap(n, slots, masks, vox), O.brickmap_scene(n, slots, masks, vox)
    top, ns, m2, v2 = O.two_level_from_bricks(n, slots, masks, vox)
    return ctx.scene_two_level(n, top, ns, m2, v2), O.two_level_scene(n, top, ns, m2, v2)


def _compare(ctx, grid, two_level, views, flags, light, what):
    sc, osc = _scenes(ctx, grid, two_level)
    hits = 0
    for k, view in enumerate(views):
        w, h = view[4], view[5]
        sh = (light, 9, 4, 9.0)
        ref = O.raymarch(osc, O.camera(*view), flags, O.shading(*sh), threads=4)
        hits += int((ref[1] < 6).sum())
        tg = R.RayTargets(ctx, w, h, index_bytes=8, counters=True)
        for count in (0, L.RAY_COUNT):  # step by step where steps are counted
            _fresh(tg)
            R.raymarch(ctx, sc, R.camera(*view), flags | count, R.shading(*sh), tg)
            ctx.sync()
            _check(ctx, tg, ref, "%s view %d" % (what, k), count=bool(count))
    sc.destroy()
    return hits


CASES = [(8, False), (40, False), (104, False), (136, False), (128, True), (256, True)]


@pytest.mark.parametrize("n,two_level", CASES)
@pytest.mark.parametrize("light", [(0.4, 1.0, 0.3), (0.0, 1.0, 0.0), (-1.0, 0.0, 0.0)])
def test_boxes_and_eyes(ctx, n, two_level, light):
    rng = np.random.default_rng(n)
    grid = np.zeros((n, n, n), np.uint16)
    lo, hi = n // 9, n - n // 5  # the box ends inside coarse blocks
    for _ in range(12):
        c = rng.integers(lo, hi, 3)
        r = int(rng.integers(1, 2 + n // 12))
        z, y, x = (slice(max(int(v) - r, 0), int(v) + r) for v in c)
        grid[z, y, x] = int(rng.integers(1, 9))
    m = n / 2.0
    views = [
        ((-0.4 * n, 1.3 * n, 1.6 * n), (m, m, m), UP, 50.0, 65, 43),
        ((float(2 * n), float(n), float(n)), (0.0, 0.0, 0.0), UP, 40.0, 33, 31),
        ((float(lo), float(hi), m), (n, 0.6 * n, 0.2 * n), UP, 90.0, 40, 40),
        ((m, float(3 * n), m), (m, 0.0, m), (0.0, 0.0, 1.0), 30.0, 1, 17),
        ((70000.0, 60000.0, m), (m, m, m), UP, 0.002 * n, 24, 24),
    ]
    hits = _compare(ctx, grid, two_level, views, L.RAY_SHADOW | L.RAY_AO, light, "n=%d" % n)
    assert hits > 0


@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("n,two_level", [(64, False), (136, False), (128, True)])
def test_cell_entered_at_the_exit(ctx, n, two_level, sign):
    # d.x equals d.z in every ray of the one pixel column, and the eye's x and
    # z differ by a whole number.  The wall ends the box in z, inside a coarse
    # block; the far voxel keeps the box open in x and y.
    gap, top, y = 2, 48, 24.0
    grid = np.zeros((n, n, n), np.uint16)
    if sign > 0:
        eye, target = (-4.5, y, -4.5 + gap), (43.5, y, 43.5 + gap)
        grid[top - 1, :, top - gap] = 7
        grid[8, 60, 60] = 3
        grid[8, 3, 3] = 3
    else:
        # towards -x, -z: the box ends at z = 8
        eye, target = (60.5, y, 60.5 - gap), (8.5, y, 8.5 - gap)
        grid[8, :, 8 + gap - 1] = 7
        grid[40, 60, 60] = 3
        grid[40, 3, 3] = 3
    view = (eye, target, UP, 50.0, 1, 65)
    assert _compare(ctx, grid, two_level, [view], L.RAY_SHADOW, (0.4, 1.0, 0.3), "exit") > 0
