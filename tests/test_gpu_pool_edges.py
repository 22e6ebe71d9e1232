"""The chunk pool's selection at the edges of its ways, against the oracle's
pool on a camera path: one load and one slot; capacities around the 256 bins
of free slots; loads around a wave, around the free bins and around the one
key per thread that the bins' way takes; both scene kinds, exact and baked
views, through filling, eviction and standing still."""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R
from tests.test_gpu_pool import PATH, _compare, _oracle_scene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scenes(ctx):
    out = {}
    for kind, gen in ((L.SCENE_TWO_LEVEL_U16, L.GEN_CAVES),
                      (L.SCENE_BRICKMAP_U16, L.GEN_HEIGHTFIELD)):
        out[kind] = (ctx.scene_generate(gen, kind, 256, 5), _oracle_scene(kind, gen, 256, 5)[0])
    yield out
    for sc, _ in out.values():
        sc.destroy()


@pytest.mark.parametrize("capacity,radius,max_loads", [
    (1, 2, 1), (2, 3, 2), (63, 4, 63), (65, 4, 64), (255, 4, 65), (256, 4, 100), (257, 6, 256),
    (512, 6, 257), (513, 7, 511), (1025, 7, 1023), (1500, 8, 1025), (1500, 12, 400)])
@pytest.mark.parametrize("kind", [L.SCENE_TWO_LEVEL_U16, L.SCENE_BRICKMAP_U16])
def test_pool_selection_edges(ctx, scenes, kind, capacity, radius, max_loads):
    sc, osc = scenes[kind]
    bake = 64 if capacity % 2 else 0
    kw = dict(capacity=capacity, quads_per_slot=64, forward_radius=radius, backward_radius=2,
              view_angle=100.0, max_loads=max_loads)
    pool = R.ChunkPool(ctx, sc, mode=L.MESH_GREEDY, bake_directions=bake, **kw)
    opool = O.OraclePool(osc, O.pool_params(greedy=True, **kw), bake_directions=bake)
    for step, (cam, fwd) in enumerate(PATH):
        pool.update(cam, fwd)
        n_cand, nl, nev, loads = opool.update(cam, fwd)
        st, g = _compare(pool, opool, step)
        assert (st["n_candidates"], st["n_loads"], st["n_evicted"]) == (n_cand, nl, nev), step
        got = np.column_stack([g["load_xyz"].reshape(-1, 3)[:nl], g["load_slot"][:nl]])
        assert np.array_equal(got, np.array(loads, np.int64).reshape(-1, 4))
    pool.destroy()
