"""Chunk edits of uploaded scenes against the oracle: masks that follow the
voxels (only the bricks a sphere reaches are touched) and masks that do not
(every brick of an edited chunk gets its mask back).  Several seeds over every
chunk, so spheres end on brick borders and reach chunk corners; the frame
afterwards reads the 2^3-block bits."""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R
from mesoengine_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,gen,n", [(L.SCENE_BRICKMAP_U16, O.GEN_TERRAIN_CAVES, 104),
                                        (L.SCENE_TWO_LEVEL_U16, O.GEN_CAVES, 128)])
@pytest.mark.parametrize("match", [True, False])
@pytest.mark.parametrize("seed", [1, 77, 4093])
def test_edit_uploaded_scene(ctx, kind, gen, n, match, seed):
    slots, masks, vox = O.build_brickmap(gen, n, 9)
    two = kind == L.SCENE_TWO_LEVEL_U16
    if two:
        top, slots, masks, vox = O.two_level_from_bricks(n, slots, masks, vox)
    masks, vox = np.ascontiguousarray(masks.copy()), np.ascontiguousarray(vox.copy())
    if not match:
        masks[1::3] = 0
    sc = (ctx.scene_two_level(n, top, slots, masks, vox) if two
          else ctx.scene_brickmap(n, slots, masks, vox))
    osc = (O.two_level_scene(n, top, slots, masks, vox) if two
           else O.brickmap_scene(n, slots, masks, vox))
    nc = -(-n // 32)
    flat = np.arange(nc ** 3)[(seed % 2)::2] if not match else np.arange(nc ** 3)
    xyz = np.stack([flat % nc, (flat // nc) % nc, flat // (nc * nc)], 1).astype(np.int32)
    dxyz = ctx.upload(xyz.ravel())
    for k in range(2):
        R.edit_chunks(sc, dxyz, len(xyz), seed + k)
        O.edit_chunks(osc, xyz, seed + k)
    a = sc.arrays()
    assert np.array_equal(a["voxels"], vox) and np.array_equal(a["masks"], masks)
    eye, target = [-0.3 * n, 1.2 * n, 0.2 * n], [0.5 * n, 0.2 * n, 0.5 * n]
    tg = R.RayTargets(ctx, 96, 64)
    flags = L.RAY_SHADOW | L.RAY_AO
    R.raymarch(ctx, sc, R.camera(eye, target, [0, 1, 0], 60.0, 96, 64), flags,
               R.shading(W.LIGHT), tg)
    ctx.sync()
    ref = O.raymarch(osc, O.camera(eye, target, [0, 1, 0], 60.0, 96, 64), flags,
                     O.shading(W.LIGHT), threads=8)
    if match:
        for got, want in zip(tg.results(), ref[:4]):
            assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    sc.destroy()
