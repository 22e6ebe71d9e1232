"""Quad visibility where quads find no room in the lists, against the oracle:
lists lowered to nothing, to less than a first lot, to a part of a shell, and to
few tests, where the largest lots are not even counted.  And what the stats say
of listed quads, of which one spans many windows of pixel tests."""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R
from mesoengine_amd import workloads as W

pytestmark = pytest.mark.gpu

W_, H_ = 320, 200
UP = [0.0, 1.0, 0.0]
# inside the caves, from outside (every chunk in one shell), just above a floor
VIEWS = {"caves": [((130.3, 140.2, 120.1), (200.0, 100.0, 180.0), 70.0),
                   ((-600.0, 500.0, -550.0), (128.0, 128.0, 128.0), 25.0)],
         "slab": [((20.0, 9.5, 6.0), (40.0, 4.0, 50.0), 70.0)]}


@pytest.fixture(scope="module")
def pools(ctx):
    out = {}
    n = 256
    caves = ctx.scene_generate(L.GEN_CAVES, L.SCENE_TWO_LEVEL_U16, n, 5)
    g = np.zeros((64, 64, 64), np.uint16)  # (z, y, x)
    g[:, :8, :] = 1
    g[20:28, 8:14, 30:40] = 2
    slab = ctx.scene_brickmap(64, *O.brickmap_from_dense(g))
    for name, sc, n, mode in [("caves", caves, 256, L.MESH_CULLED), ("slab", slab, 64, L.MESH_GREEDY)]:
        nc = n // 32
        pool = R.ChunkPool(ctx, sc, capacity=nc ** 3, quads_per_slot=16384, forward_radius=16,
                           backward_radius=16, view_angle=120.0, max_loads=nc ** 3, mode=mode)
        pool.update((nc // 2,) * 3, (1.0, 0.0, 0.0))
        out[name] = (n, nc, pool, pool.state())
    yield out
    for _, _, pool, _ in out.values():
        pool.destroy()
    caves.destroy()
    slab.destroy()


def _draw(ctx, pools, name, view, limits):
    n, nc, pool, st = pools[name]
    eye, target, fov = view
    rast = R.Raster(ctx, W_, H_)
    if limits:
        L.check(ctx.lib.meso_raster_set_list_limits(rast.h, *limits))
    tg = R.RayTargets(ctx, W_, H_)
    for b in (tg.index, tg.face, tg.t, tg.shade):
        b.fill(0xA5)
    for _ in range(2):  # a second frame starts from what the first one left
        rast.draw(pool, R.camera(eye, target, UP, fov, W_, H_), R.shading(W.LIGHT), tg)
    ctx.sync()
    stats = rast.stats()
    ref = O.raster_pool(O.camera(eye, target, UP, fov, W_, H_), n, nc, st["slot_chunk"],
                        st["slot_count"], st["quads"], 16384, O.shading(W.LIGHT).light)
    for got, want in zip(tg.results(), ref[:4]):
        assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), (name, limits)
    rast.destroy()
    return stats


LIMITS = [(0, 0), (1, 1 << 23), (300, 1 << 23), (20_000, 1 << 23), (1 << 22, 1), (1 << 22, 400)]


@pytest.mark.parametrize("limits", LIMITS)
@pytest.mark.parametrize("name,k", [("caves", 0), ("caves", 1), ("slab", 0)])
def test_quads_without_room(ctx, pools, name, k, limits):
    free = _draw(ctx, pools, name, VIEWS[name][k], None)
    assert free["overflow_quads"] == 0
    stats = _draw(ctx, pools, name, VIEWS[name][k], limits)
    assert stats["segments"] + stats["overflow_quads"] == stats["small_quads"] + stats["large_quads"]
    if name == "caves" and limits != (20_000, 1 << 23):
        assert stats["overflow_quads"] > 0
    if name == "caves" and k == 1:  # far more quads than lots listed before the lists are full
        assert stats["overflow_quads"] > 20 * 1024


def test_listed_quads(ctx, pools):
    # the floor's quads cover thousands of pixels: many windows of 256 tests each
    stats = _draw(ctx, pools, "slab", VIEWS["slab"][0], None)
    assert stats["large_quads"] > 0 and stats["overflow_quads"] == 0
    assert stats["segments"] == stats["small_quads"] + stats["large_quads"]
    n, nc, pool, st = pools["slab"]
    eye, target, fov = VIEWS["slab"][0]
    ref = O.raster_pool(O.camera(eye, target, UP, fov, W_, H_), n, nc, st["slot_chunk"],
                        st["slot_count"], st["quads"], 16384, O.shading(W.LIGHT).light)
    top = ref[0][ref[1] == 2]  # +y hits: of the four 32x32 floor quads at least one is so large
    assert len(top) // 4 > 4 * 256


# quads of more pixels than a quad has tests, and a frame above the 2^26 pixels
# up to which a test is one pixel
@pytest.mark.parametrize("w,h", [(1920, 1080), (16384, 4097)])
def test_quads_of_many_pixels(ctx, pools, w, h):
    n, nc, pool, st = pools["slab"]
    eye, target, fov = (20.3, 9.1, 6.2), (40.0, 4.0, 50.0), 70.0
    rast, tg = R.Raster(ctx, w, h), R.RayTargets(ctx, w, h)
    rast.draw(pool, R.camera(eye, target, UP, fov, w, h), R.shading(W.LIGHT), tg)
    ctx.sync()
    assert rast.stats()["overflow_quads"] == 0
    ref = O.raster_pool(O.camera(eye, target, UP, fov, w, h), n, nc, st["slot_chunk"],
                        st["slot_count"], st["quads"], 16384, O.shading(W.LIGHT).light)
    assert (ref[1] == 2).sum() > 1 << 19  # the floor's few quads
    for got, want in zip(tg.results(), ref[:4]):
        assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    rast.destroy()
