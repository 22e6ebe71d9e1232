"""Eyes so far off that rounding puts hit points, and with them the origins of
shadow and occlusion rays, outside the scene, against the oracle.

Dense: frames whose pixels are a few thousandths of a voxel and less, at the
edge of a slab at either end of the grid, with the light toward that end, so
that shadow rays start beyond the plane they leave by (counted on the CPU).
The default launch, 8x8 tiles (four lanes a ray both) and 16x16 tiles.
"""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R

from test_gpu_variants import _check, _force, _fresh

pytestmark = pytest.mark.gpu


def _beyond(ocam, ref, n, light):
    """Lit hits whose point lies outside the grid on a side that the light is toward."""
    w = ocam.width
    count = 0
    for pix in np.flatnonzero(ref[1] < 6):
        f = int(ref[1][pix])
        axis = 2 - f // 2
        sign = -1 if f & 1 else 1
        if light[axis] * sign <= 0:
            continue
        o, d = O.primary_ray(ocam, int(pix % w), int(pix // w))
        p = o + d * ref[2][pix]
        i = int(ref[0][pix])
        start = [i % n, i // n % n, i // n // n]
        start[axis] += sign
        if all(0 <= c < n for c in start):
            count += any((p[a] < 0 and light[a] < 0) or (p[a] > n and light[a] > 0)
                         for a in range(3))
    return count


def dense_edge(n, axis, up_axis, high, dist, rng):
    """A slab up to the middle of `up_axis`, an eye and a light for its edge at the
    low or high end of `axis`."""
    sl = [slice(None)] * 3
    sl[2 - up_axis] = slice(0, n // 2)
    grid = np.zeros((n, n, n), np.uint8)  # (z, y, x)
    grid[tuple(sl)] = 2
    target, direction, light = [n * 0.43] * 3, [0.17] * 3, [0.11] * 3
    target[axis], target[up_axis] = (n if high else 0.0), n // 2
    direction[axis], direction[up_axis] = (-0.6 if high else 0.6), 0.7
    light[axis], light[up_axis] = (0.6 if high else -0.6), 0.8
    eye = [float(np.float32(t + dist * (c + 0.3 * (j - 0.5))))
           for t, c, j in zip(target, direction, rng.random(3))]
    up = [0.0, 0.0, 0.0]
    up[3 - axis - up_axis] = 1.0
    return grid, eye, target, up, light


# a hit point lies beyond a side when its plane and the side's plane are crossed
# at one t, where the axes' order enters the voxel first: axis after up_axis
@pytest.mark.parametrize("dist", [3000.0, 60000.0])
@pytest.mark.parametrize("high", [0, 1])
@pytest.mark.parametrize("axis,up_axis", [(1, 0), (2, 0), (2, 1)])
@pytest.mark.parametrize("n", [16, 63])
def test_dense_shadow_rays_from_beyond_the_grid(ctx, tmp_path, n, axis, up_axis, high, dist):
    rng = np.random.default_rng(7)
    w, h, flags, beyond = 57, 41, L.RAY_SHADOW, 0
    fov = float(np.degrees(300 * 2.0 ** -24 * h))  # some 300 roundings of the distance a pixel
    tg = R.RayTargets(ctx, w, h)
    for frame in range(8):
        grid, eye, target, up, light = dense_edge(n, axis, up_axis, high, dist, rng)
        view = (eye, target, up, fov, w, h)
        ocam, sh = O.camera(*view), (light, 3, 4, 5.0)
        ref = O.raymarch(O.dense_scene(grid.ravel()), ocam, flags, O.shading(*sh), threads=4)
        beyond += _beyond(ocam, ref, n, light)
        sc = ctx.scene_dense(grid)
        for shape in [None, (0, 16, 16, 0), (2, 8, 8, 0)]:
            if shape:
                _force(ctx, tmp_path, L.SCENE_DENSE_U8, n, w, h, flags, shape)
            _fresh(tg)
            R.raymarch(ctx, sc, R.camera(*view), flags, R.shading(*sh), tg)
            ctx.sync()
            _check(ctx, tg, ref, "n=%d axis %d %s" % (n, axis, shape), count=False)
        sc.destroy()
    assert beyond > 0


# An eye 2^46 voxels away and more: the few directions that hit the scene put
# the hit point millions of voxels off, also along an axis that the light has no
# part in, on which shadow rays then do not move (counted on the CPU).
@pytest.mark.parametrize("kind", [L.SCENE_BRICKMAP_U16, L.SCENE_TWO_LEVEL_U16])
def test_brick_shadow_rays_from_far_off_an_axis(ctx, kind):
    n, w, h, flags = 128, 9, 8, L.RAY_SHADOW | L.RAY_AO
    grid = np.zeros((n, n, n), np.uint16)
    grid[np.random.default_rng(3).random((n, n, n)) < 0.2] = 3
    bricks = O.brickmap_from_dense(grid)
    if kind == L.SCENE_BRICKMAP_U16:
        sc, osc = ctx.scene_brickmap(n, *bricks), O.brickmap_scene(n, *bricks)
    else:
        nodes = O.two_level_from_bricks(n, *bricks)
        sc, osc = ctx.scene_two_level(n, *nodes), O.two_level_scene(n, *nodes)
    tg = R.RayTargets(ctx, w, h, index_bytes=8)
    far = 0
    for e, seed in [(e, seed) for e in (46, 50, 52) for seed in range(30)]:
        d = np.random.default_rng(seed).normal(size=3)
        eye = [float(np.float32(c * 2.0 ** e)) for c in d / np.linalg.norm(d)]
        view = (eye, (n / 2.0,) * 3, (0.1, 1.0, 0.2), 1e-6, w, h)
        ocam = O.camera(*view)
        for light in [(0.0, 1.0, 0.0), (1.0, 0.0, 0.0), (0.0, 0.0, -1.0), (0.0, -1.0, 0.0)]:
            ref = O.raymarch(osc, ocam, flags, O.shading(light, 1, 4, 5.0))
            hits = np.flatnonzero(ref[1] < 6)
            if not len(hits):
                break
            for pix in hits:
                o, dd = O.primary_ray(ocam, int(pix % w), int(pix // w))
                p = o + dd * ref[2][pix]
                axis, sign = 2 - ref[1][pix] // 2, -1 if ref[1][pix] & 1 else 1
                far += light[axis] * sign > 0 and any(light[a] == 0 and p[a] > 2 ** 20 + n
                                                      for a in range(3))
            _fresh(tg)
            R.raymarch(ctx, sc, R.camera(*view), flags, R.shading(light, 1, 4, 5.0), tg)
            ctx.sync()
            _check(ctx, tg, ref, "2^%d seed %d light %s" % (e, seed, light), count=False)
    sc.destroy()
    assert far > 0


# An eye whose squared distance is above the largest float, looking along x: one
# ray hits a slab's side all the same.  And one just below it.
@pytest.mark.parametrize("dist", [1e18, 1.8e19, 1e20, 3e38])
def test_quads_seen_from_beyond_the_squares(ctx, dist):
    g = np.zeros((64, 64, 64), np.uint16)  # (z, y, x)
    g[:, :8, :] = 1
    sc = ctx.scene_brickmap(64, *O.brickmap_from_dense(g))
    pool = R.ChunkPool(ctx, sc, capacity=8, quads_per_slot=1024, forward_radius=4,
                       backward_radius=4, view_angle=120.0, max_loads=8)
    pool.update((1, 1, 1), (1.0, 0.0, 0.0))
    st = pool.state()
    rast, tg = R.Raster(ctx, 3, 3), R.RayTargets(ctx, 1, 1)
    eye = (float(np.float32(dist)), 4.5, 20.5)
    view = (eye, (eye[0] * 0.999, 4.5, 20.5), (0.0, 1.0, 0.0), 40.0, 1, 1)
    ref = O.raster_pool(O.camera(*view), 64, 2, st["slot_chunk"], st["slot_count"], st["quads"], 1024,
                        O.shading((0.5, 1.0, 0.3)).light)
    assert (ref[1][0] == 4) == (dist < 1e38)  # (at 3e38 the camera has no direction)
    rast.draw(pool, R.camera(*view), R.shading((0.5, 1.0, 0.3)), tg)
    ctx.sync()
    for got, want in zip(tg.results(), ref[:4]):
        assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    rast.destroy()
    pool.destroy()
    sc.destroy()
