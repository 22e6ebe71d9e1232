"""Taking a served result: the block is staged in chunks of 2 MiB and shared
out over threads.

Frames below, at and just over the ends of a chunk, arrays that end on one and
inside one, subsets of the arrays with gaps between them, 8-byte indices, and
several threads taking at once, each against the plain path's arrays.
"""
import ctypes as C
import threading

import numpy as np
import pytest

from mesoengine_amd import _lib as L
from mesoengine_amd import runtime as R
from mesoengine_amd import workloads as W

pytestmark = pytest.mark.gpu

PARTS = ("index", "face", "t", "shade")
# 13 bytes a pixel: 161202 pixels are just below 2 MiB, 161334 above; 1024 x 512 has an index
# array of exactly 2 MiB, 2048 x 1024 a face array too
SIZES = [(1, 1), (37, 3), (401, 402), (8963, 18), (1024, 512), (1025, 511), (2048, 1024), (1500, 901)]


@pytest.fixture(scope="module")
def setup(ctx):
    sc = ctx.scene_generate(L.GEN_TERRAIN_CAVES, L.SCENE_BRICKMAP_U16, 128, 3)
    srv = R.Server(ctx, 256 << 20, max_pending=64, max_inflight=16, idle_exit_us=2000)
    yield sc, srv
    srv.stop()
    sc.destroy()


def _cam(n, w, h):
    return R.camera([1.6 * n, 1.3 * n, 1.5 * n], [n / 2, n * 0.2, n / 2], [0.0, 1.0, 0.0], 55.0, w, h)


def _plain(ctx, sc, w, h, index_bytes=4):
    tg = R.RayTargets(ctx, w, h, index_bytes=index_bytes)
    R.raymarch(ctx, sc, _cam(sc.info().n, w, h), L.RAY_SHADOW, R.shading(W.LIGHT), tg)
    ctx.sync()
    return tg.results()


def _served(srv, sc, w, h, index_bytes=4, parts=PARTS):
    tk = srv.submit(sc, _cam(sc.info().n, w, h), L.RAY_SHADOW, R.shading(W.LIGHT))
    srv.wait(tk, 30_000_000)
    return srv.take(tk, w, h, index_bytes, parts)


def _same(got, ref, parts=PARTS):
    for name, a, b in zip(PARTS, got, ref):
        if name not in parts:
            assert a is None
            continue
        assert a.dtype == b.dtype and np.array_equal(a.view(np.uint8), b.view(np.uint8)), name


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "%dx%d" % s)
def test_whole_results(ctx, setup, size):
    sc, srv = setup
    ref = _plain(ctx, sc, *size)
    assert ref[0].dtype == np.int64
    for index_bytes in (4, 0):
        _same(_served(srv, sc, *size, index_bytes), ref)
    # the entry without the widening, and a size it doesn't hold
    w, h = size
    tk = srv.submit(sc, _cam(128, w, h), L.RAY_SHADOW, R.shading(W.LIGHT))
    srv.wait(tk, 30_000_000)
    with pytest.raises(L.MesoError):
        srv.take(tk, w, h, 8)
    arr = [np.empty(w * h, d) for d in (np.int32, np.uint8, np.float32, np.float32)]
    o = L.HostOutputs(C.sizeof(L.HostOutputs), 4, *[a.ctypes.data for a in arr])
    L.check(ctx.lib.meso_serve_take(srv.h, tk, C.byref(o)))
    _same([arr[0].astype(np.int64)] + arr[1:], ref)


@pytest.mark.parametrize("parts", [("face",), ("index", "shade"), ("face", "t"), ("t",),
                                   ("index", "face", "shade")])
def test_some_arrays(ctx, setup, parts):
    sc, srv = setup
    for size in [(64, 5), (513, 511), (1500, 901)]:
        _same(_served(srv, sc, *size, 4, parts), _plain(ctx, sc, *size), parts)


def test_wide_indices(ctx, setup):
    _, srv = setup
    sc = ctx.scene_generate(L.GEN_HEIGHTFIELD, L.SCENE_TWO_LEVEL_U16, 1408, 5)
    for size in [(7, 9), (700, 601)]:
        ref = _plain(ctx, sc, *size, index_bytes=8)
        for index_bytes in (8, 0):
            _same(_served(srv, sc, *size, index_bytes), ref)
    sc.destroy()


@pytest.mark.parametrize("n", [5, 16, 61])
def test_dense_scenes(ctx, setup, n):
    _, srv = setup
    sc = ctx.scene_generate(L.GEN_SPHERES, L.SCENE_DENSE_U8, n, 2, 5)
    for size in [(1, 1), (123, 77), (640, 361)]:
        _same(_served(srv, sc, *size), _plain(ctx, sc, *size))
    sc.destroy()


def test_threads_take_at_once(ctx, setup):
    sc, srv = setup
    sizes = [(1500, 901), (1201, 700), (64, 64)]
    refs = [_plain(ctx, sc, *s) for s in sizes]
    errors = []

    def take(k):
        try:
            for _ in range(4):
                _same(_served(srv, sc, *sizes[k]), refs[k])
        except BaseException as e:  # surfaced after the join
            errors.append(e)

    threads = [threading.Thread(target=take, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
