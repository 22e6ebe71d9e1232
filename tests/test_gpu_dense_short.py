"""Rays of dense grids that end within a few cells, against the oracle: solid
grids, rough ones of many fills, eyes inside and on the sides, short occlusion
rays; frames whose rays four lanes walk, up to the line (two 8x8 waves per SIMD
of 256 CUs) and a column past it, 16x16 tiles, and served frames."""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R

from test_gpu_variants import _check, _force, _fresh

pytestmark = pytest.mark.gpu

UP = (0.0, 1.0, 0.0)
LIGHT = (-0.4, 0.9, 0.3)


def _compare(ctx, tmp_path, grid, view, radius, server=None):
    n, (w, h) = grid.shape[0], view[4:]
    flags = L.RAY_SHADOW | L.RAY_AO
    sc, osc = ctx.scene_dense(grid), O.dense_scene(grid.ravel())
    sh = (LIGHT, 5, 3, radius)
    ref = O.raymarch(osc, O.camera(*view), flags, O.shading(*sh), threads=4)
    tg = R.RayTargets(ctx, w, h)
    for shape in [(2, 8, 8, 0), (0, 16, 16, 0), (5, 8, 8, 0)]:  # the first: the default
        _force(ctx, tmp_path, L.SCENE_DENSE_U8, n, w, h, flags, shape)
        _fresh(tg)
        R.raymarch(ctx, sc, R.camera(*view), flags, R.shading(*sh), tg)
        ctx.sync()
        _check(ctx, tg, ref, "n=%d %s %s" % (n, view, shape), count=False)
    if server:
        tk = server.submit(sc, R.camera(*view), flags, R.shading(*sh))
        server.wait(tk, 30_000_000)
        for got, want in zip(server.take(tk, w, h), ref[:4]):
            assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    sc.destroy()


@pytest.mark.parametrize("n", [3, 9, 23, 40])
@pytest.mark.parametrize("fill", [0.02, 0.1, 0.5, 0.9, 1.0])
def test_fills_and_eyes(ctx, tmp_path, n, fill):
    rng = np.random.default_rng(n)
    grid = (rng.random((n, n, n)) < fill).astype(np.uint8) * 3
    m = n / 2.0
    server = R.Server(ctx, 64 << 20, max_pending=8, max_inflight=8, idle_exit_us=2000)
    for k, view in enumerate([((-0.4 * n, 1.3 * n, 1.6 * n), (m, m, m), UP, 50.0),
                              ((m + 0.25, 0.6 * n, m), (n, 0.1 * n, 0.2 * n), UP, 90.0),
                              ((m, float(n), m), (0.0, 0.0, 0.0), UP, 80.0),
                              ((m, 0.5 * n, 0.0), (m, 0.5 * n, float(n)), UP, 100.0)]):
        size = [(53, 37), (96, 95), (31, 62), (40, 41)][k]
        _compare(ctx, tmp_path, grid, view + size, (3.5, 0.7, 20.0, 8.0)[k], server)
    server.stop()


@pytest.mark.parametrize("size", [(512, 256), (513, 256), (8, 16384), (1, 1)])
def test_the_line(ctx, tmp_path, size):
    grid = (np.random.default_rng(1).random((24, 24, 24)) < 0.2).astype(np.uint8)
    _compare(ctx, tmp_path, grid, ((37.0, 30.0, 33.0), (11.0, 12.0, 13.0), UP, 55.0) + size, 4.0)
