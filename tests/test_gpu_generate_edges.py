"""Generated scenes at the edges of the voxelization kernels' ranges, against
the oracle: one brick; edges that end inside a 32^3 block; noise cells smaller
than a brick (hashed per voxel), exactly one brick, and wider ones that
straddle bricks; a node's worth of bricks; more bricks than one pass of waves.
Slots, masks, voxels and the solid count are equal, and a small frame (which
reads the empty-space levels and the solid box) is the same bits."""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R
from mesoengine_amd import workloads as W

pytestmark = pytest.mark.gpu

CASES = [(O.GEN_TERRAIN_CAVES, n) for n in (8, 24, 40, 104, 128, 200, 256, 264, 296)] + \
        [(O.GEN_HEIGHTFIELD, n) for n in (8, 72, 136)] + \
        [(O.GEN_CAVES, n) for n in (8, 40, 128, 168)]


@pytest.mark.parametrize("gen,n", CASES)
@pytest.mark.parametrize("two_level", [False, True])
def test_generated_scene_edges(ctx, gen, n, two_level):
    if two_level and n % 128:
        n = 128
    seed = 1000 + n
    layout = L.SCENE_TWO_LEVEL_U16 if two_level else L.SCENE_BRICKMAP_U16
    sc = ctx.scene_generate(gen, layout, n, seed)
    a = sc.arrays()
    slots, masks, vox = O.build_brickmap(gen, n, seed)
    if two_level:
        top, slots, masks, vox = O.two_level_from_bricks(n, slots, masks, vox)
        assert np.array_equal(a["top"], top)
        osc = O.two_level_scene(n, top, slots, masks, vox)
    else:
        osc = O.brickmap_scene(n, slots, masks, vox)
    assert np.array_equal(a["slots"], slots.ravel())
    assert np.array_equal(a["masks"], masks)
    assert np.array_equal(a["voxels"], vox)
    assert sc.info().solid_voxels == int((vox != 0).sum())
    eye, target = [-0.4 * n, 1.1 * n, 0.3 * n], [0.6 * n, 0.2 * n, 0.5 * n]
    up, w, h = [0.0, 1.0, 0.0], 61, 37
    tg = R.RayTargets(ctx, w, h)
    R.raymarch(ctx, sc, R.camera(eye, target, up, 60.0, w, h), L.RAY_SHADOW | L.RAY_AO,
               R.shading(W.LIGHT), tg)
    ctx.sync()
    ref = O.raymarch(osc, O.camera(eye, target, up, 60.0, w, h), O.RAY_SHADOW | O.RAY_AO,
                     O.shading(W.LIGHT), threads=8)
    for got, want in zip(tg.results(), ref[:4]):
        assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    sc.destroy()
