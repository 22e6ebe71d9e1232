"""Quad visibility at the edges of its splits, against the oracle: frames of one
pixel, of less than a block of 8, 32 or 128 pixels and one more; eyes inside
the volume, where nearer chunks hide farther ones and quads reach behind the
eye; an eye just above a surface; narrow and very wide views; a pool whose
slots cut their meshes short."""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R
from mesoengine_amd import workloads as W

pytestmark = pytest.mark.gpu

FRAMES = [(1, 1), (7, 3), (8, 8), (33, 9), (31, 129), (129, 130), (257, 64)]
VIEWS = [((130.3, 140.2, 120.1), (200.0, 100.0, 180.0), 70.0),
         ((20.5, 250.0, 30.0), (128.0, 90.0, 128.0), 20.0),
         ((128.0, 128.0, 128.0), (128.5, 100.0, 129.0), 150.0),
         ((64.01, 65.02, 64.5), (66.0, 64.0, 90.0), 100.0)]


@pytest.fixture(scope="module")
def caves(ctx):
    n = 256
    sc = ctx.scene_generate(L.GEN_CAVES, L.SCENE_TWO_LEVEL_U16, n, 5)
    pools = []
    for per in (65536, 900):
        pool = R.ChunkPool(ctx, sc, capacity=512, quads_per_slot=per, forward_radius=16,
                           backward_radius=16, view_angle=120.0, max_loads=512)
        pool.update((4, 4, 4), (1.0, 0.0, 0.0))
        pools.append((pool, per, pool.state()))
    yield n, pools
    for pool, _, _ in pools:
        pool.destroy()
    sc.destroy()


@pytest.mark.parametrize("w,h", FRAMES)
@pytest.mark.parametrize("eye,target,fov", VIEWS)
def test_raster_edges_match_oracle(ctx, caves, w, h, eye, target, fov):
    n, pools = caves
    rast = R.Raster(ctx, 257, 130)
    tg = R.RayTargets(ctx, w, h)
    sh = R.shading(W.LIGHT)
    up = [0.0, 1.0, 0.0]
    for pool, per, st in pools:
        rast.draw(pool, R.camera(eye, target, up, fov, w, h), sh, tg)
        ctx.sync()
        ref = O.raster_pool(O.camera(eye, target, up, fov, w, h), n, 8, st["slot_chunk"],
                            st["slot_count"], st["quads"], per, O.shading(W.LIGHT).light)
        for got, want in zip(tg.results(), ref[:4]):
            assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    rast.destroy()
