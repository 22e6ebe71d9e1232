"""Quad visibility drawn in shells and in one go, against the oracle: which one
a frame takes goes by its resident chunks and pixels, and the line between them
is moved here so that frames of every size take both, with room in the lists
and without."""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R
from mesoengine_amd import workloads as W

from test_gpu_raster_edges import FRAMES, VIEWS, caves  # noqa: F401

pytestmark = pytest.mark.gpu

UP = [0.0, 1.0, 0.0]


@pytest.mark.parametrize("w,h", FRAMES + [(640, 360)])
@pytest.mark.parametrize("eye,target,fov", VIEWS)
def test_shells_match_oracle(ctx, caves, w, h, eye, target, fov):  # noqa: F811
    n, pools = caves
    rast = R.Raster(ctx, 640, 360)
    tg = R.RayTargets(ctx, w, h)
    sh = R.shading(W.LIGHT)
    for pool, per, st in pools:
        ref = O.raster_pool(O.camera(eye, target, UP, fov, w, h), n, 8, st["slot_chunk"],
                            st["slot_count"], st["quads"], per, O.shading(W.LIGHT).light)
        drawn = []
        for line, records in [(0, 1 << 22), (1 << 63, 1 << 22), (0, 2000)]:
            L.check(ctx.lib.meso_raster_set_shell_line(rast.h, line))
            L.check(ctx.lib.meso_raster_set_list_limits(rast.h, records, 1 << 23))
            for b in (tg.index, tg.face, tg.t, tg.shade):
                b.fill(0xA5)
            rast.draw(pool, R.camera(eye, target, UP, fov, w, h), sh, tg)
            ctx.sync()
            for got, want in zip(tg.results(), ref[:4]):
                assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), (line, records)
            s = rast.stats()
            assert s["segments"] + s["overflow_quads"] == s["small_quads"] + s["large_quads"]
            drawn.append(s["segments"] + s["overflow_quads"])
        # the shells leave hidden quads out, whatever the lists hold
        assert drawn[0] <= drawn[1] and drawn[2] == drawn[0]
    rast.destroy()


def test_default_line(ctx, caves):  # noqa: F811
    # 512 chunks: one go up to 2^23 pixels, shells above
    _, pools = caves
    pool = pools[0][0]
    eye, target, fov = VIEWS[0]
    counts = {}
    for w, h in [(4096, 2048), (4096, 2049)]:
        rast, tg = R.Raster(ctx, w, h), R.RayTargets(ctx, w, h)
        for line in (None, 0, 1 << 63):
            if line is not None:
                L.check(ctx.lib.meso_raster_set_shell_line(rast.h, line))
            rast.draw(pool, R.camera(eye, target, UP, fov, w, h), R.shading(W.LIGHT), tg)
            counts[h, line] = rast.stats()["segments"]
        rast.destroy()
    assert counts[2048, None] == counts[2048, 1 << 63] > counts[2048, 0]
    assert counts[2049, None] == counts[2049, 0] < counts[2049, 1 << 63]
