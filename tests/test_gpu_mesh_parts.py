"""Batches of fewer chunks than CUs, whose quads several workgroups write:
batch lengths where the number of workgroups per chunk changes (256 CUs), and
a batch capacity that ends inside a chunk, against the oracle."""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R

pytestmark = pytest.mark.gpu


def _chunks():
    z, y, x = np.indices((32, 32, 32))
    rng = np.random.default_rng(23)
    one = np.zeros((32, 32, 32), int)
    one[0, 31, 7] = 2
    return [np.zeros((32, 32, 32), int), one, (x + y + z) % 2, 1 + (z // 3) % 5,
            np.where(rng.random((32, 32, 32)) < 0.4, rng.integers(1, 4, (32, 32, 32)), 0)]


@pytest.mark.parametrize("n", [1, 2, 64, 65, 85, 86, 128, 129, 256, 257])
@pytest.mark.parametrize("mode", [L.MESH_CULLED, L.MESH_GREEDY])
def test_batches_at_the_splits(ctx, n, mode):
    kinds = _chunks()
    ref = [O.mesh_chunk(k.astype(np.uint16).ravel(), mode == L.MESH_GREEDY) for k in kinds]
    pick = np.random.default_rng(n).integers(0, len(kinds), n)
    pick[0] = 2 if n == 1 else pick[0]
    buf = ctx.upload(np.stack([kinds[k] for k in pick]).astype(np.uint16))
    want = np.concatenate([ref[k] for k in pick])
    for cap in sorted({len(want), max(len(want) // 2 + 13, 1)}):
        mt = R.MeshTargets(ctx, n, cap)
        mt.quads.fill(0xEE)
        R.mesh_chunks(ctx, R.chunk_source(buf, 2, n), mode, mt)
        ctx.sync()
        counts, prefix, total, quads = mt.results()
        assert np.array_equal(counts, [len(ref[k]) for k in pick])
        assert np.array_equal(prefix, np.concatenate([[0], np.cumsum(counts)[:-1]]))
        assert total == len(want)
        assert np.array_equal(quads, want[:cap])
