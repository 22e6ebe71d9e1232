"""Every pixel of a frame is traced once, whatever its shape.

The tiled launches hand groups of tiles to the XCDs, cut by the number of tile
rows: frames of one pixel, of one row and one column, and at the edges of the
two row counts at which the cut changes (24 and 64 rows of 8, and of 16).
"""
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R

from test_gpu_variants import _check, _force, _fresh

pytestmark = pytest.mark.gpu

N = 40
LIGHT = (0.4, 1.0, 0.3)
FRAMES = [(1, 1), (9, 7), (1, 515), (907, 1), (2001, 9), (57, 184), (58, 185), (7, 369), (33, 504),
          (65, 505), (17, 1025)]


@pytest.mark.parametrize("size", FRAMES, ids=lambda s: "%dx%d" % s)
def test_every_pixel_of_the_frame(ctx, tmp_path, size):
    w, h = size
    sc = ctx.scene_generate(L.GEN_SPHERES, L.SCENE_DENSE_U8, N, 1, 4)
    view = ([55.0, 47.0, 51.0], [18.0, 20.0, 21.0], [0.0, 1.0, 0.0], 60.0, w, h)
    cam = R.camera(*view)
    osc = O.dense_scene(O.spheres_dense(1, N, 4).ravel())
    ocam = O.camera(*view)
    ref = O.raymarch(osc, ocam, O.RAY_SHADOW, O.shading(LIGHT), threads=4)
    tg = R.RayTargets(ctx, w, h)
    # no shape tuned, then each tiled shape
    for shape in [None, (0, 16, 16, 0), (1, 32, 8, 0), (2, 8, 8, 0), (3, 16, 8, 0), (4, 32, 16, 0)]:
        if shape:
            _force(ctx, tmp_path, L.SCENE_DENSE_U8, N, w, h, L.RAY_SHADOW, shape)
        _fresh(tg)
        R.raymarch(ctx, sc, cam, L.RAY_SHADOW, R.shading(LIGHT), tg)
        ctx.sync()
        _check(ctx, tg, ref, "%dx%d %s" % (w, h, shape), count=False)
    sc.destroy()
