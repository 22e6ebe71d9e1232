"""Chunk meshing at the edges of the emission's splits, against the oracle:
no quad, one quad, a row of 32 quads ending at once, quad lists of one window
less and more, the most quads a chunk can have, tall and wide quads, and
capacities that cut the output inside a window.  u8 and u16, culled and
greedy, one chunk alone and all in one batch."""
import numpy as np
import pytest

import oracle as O
from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R

pytestmark = pytest.mark.gpu


def _chunks():
    z, y, x = np.indices((32, 32, 32))
    rng = np.random.default_rng(17)
    out = [np.zeros((32, 32, 32), int), np.ones((32, 32, 32), int)]
    one = np.zeros((32, 32, 32), int)
    one[31, 31, 31] = 3
    out.append(one)
    out.append((x + y + z) % 2)                   # 98,304 quads of one face
    out.append((x % 2) * (1 + y // 16))           # columns: 32 quads end in one row
    out.append(((x + z) % 2) * (y < 20))
    out.append(1 + (z // 3) % 5)                  # wide slabs of materials
    out.append(np.where(rng.random((32, 32, 32)) < 0.5, rng.integers(1, 4, (32, 32, 32)), 0))
    for count in (671, 672, 673, 1343, 1344, 1345):  # 6 quads each: around 4032 and 8064
        g = np.zeros(32768, int)
        free = np.flatnonzero(((x % 2) | (y % 2) | (z % 2)).ravel() == 0)
        g[rng.permutation(free)[:count]] = 1
        out.append(g.reshape(32, 32, 32))
    out.append(np.where((x // 8 + y // 8 + z // 8) % 2, 1 + x // 16, 0))
    return np.stack(out)


@pytest.mark.parametrize("elem", [1, 2])
@pytest.mark.parametrize("mode", [L.MESH_CULLED, L.MESH_GREEDY])
def test_mesh_edges_match_oracle(ctx, elem, mode):
    vox = _chunks()
    n = len(vox)
    ref = [O.mesh_chunk(v.astype(np.uint16).ravel(), mode == L.MESH_GREEDY) for v in vox]
    buf = ctx.upload(vox.astype(np.uint8 if elem == 1 else np.uint16))
    cnt, q = ctx.buffer(4), ctx.buffer(4 * 98304)
    for c in range(n):
        for cap in sorted({98304, len(ref[c]), len(ref[c]) // 2, min(len(ref[c]), 4033), 1}):
            q.fill(0xEE)
            R.mesh_chunk(ctx, buf.ptr + c * 32768 * elem, elem, mode, cnt.ptr, q.ptr, cap)
            ctx.sync()
            assert int(cnt.download(np.uint32)[0]) == len(ref[c])
            got = q.download(np.uint32)
            k = min(cap, len(ref[c]))
            assert np.array_equal(got[:k], ref[c][:k])
            assert (got[k:] == 0xEEEEEEEE).all()
    mt = R.MeshTargets(ctx, n, sum(len(r) for r in ref))
    R.mesh_chunks(ctx, R.chunk_source(buf, elem, n), mode, mt)
    ctx.sync()
    counts, prefix, total, quads = mt.results()
    assert np.array_equal(counts, [len(r) for r in ref])
    assert np.array_equal(prefix, np.concatenate([[0], np.cumsum(counts)[:-1]]))
    assert total == mt.capacity and np.array_equal(quads, np.concatenate(ref))
