"""Taking a served result into pinned memory (meso_host_alloc), which is copied
to straight: all arrays pinned, some of them, arrays inside one allocation, both
take entries, and several threads at once, each against the plain path."""
import ctypes as C
import threading

import numpy as np
import pytest

from mesoengine_amd import _lib as L

from test_gpu_serving_take import _cam, _plain, _same, setup  # noqa: F401
from mesoengine_amd import runtime as R
from mesoengine_amd import workloads as W

pytestmark = pytest.mark.gpu

DTYPES = (np.int32, np.uint8, np.float32, np.float32)


class _Pinned:
    def __init__(self, ctx, nbytes):
        self.ctx, p = ctx, C.c_void_p()
        L.check(ctx.lib.meso_host_alloc(ctx.h, nbytes, C.byref(p)))
        self.ptr, self.nbytes = p.value, nbytes
        self.bytes = np.ctypeslib.as_array((C.c_uint8 * nbytes).from_address(self.ptr))
        self.bytes[:] = 0xA5

    def array(self, at, dtype, n):
        return self.bytes[at:at + n * np.dtype(dtype).itemsize].view(dtype)

    def free(self):
        L.check(self.ctx.lib.meso_host_free(self.ctx.h, self.ptr))


def _take(ctx, srv, sc, size, pinned, wide):
    """pinned: which of the four arrays; the others are ordinary memory"""
    w, h = size
    n = w * h
    dtypes = ((np.int64,) if wide else (np.int32,)) + DTYPES[1:]
    mem = _Pinned(ctx, 64 + 8 * n + 16 * n)
    arrays, at = [], 16
    for k, d in enumerate(dtypes):
        arrays.append(mem.array(at, d, n) if k in pinned else np.full(n, 7, d))
        at += -(-n * np.dtype(d).itemsize // 16) * 16
    tk = srv.submit(sc, _cam(128, w, h), L.RAY_SHADOW, R.shading(W.LIGHT))
    srv.wait(tk, 30_000_000)
    o = L.HostOutputs(C.sizeof(L.HostOutputs), 4, *[a.ctypes.data for a in arrays])
    entry = ctx.lib.meso_serve_take_wide if wide else ctx.lib.meso_serve_take
    L.check(entry(srv.h, tk, C.byref(o)))
    got = [arrays[0].astype(np.int64)] + [a.copy() for a in arrays[1:]]
    assert (mem.bytes[:16] == 0xA5).all()
    mem.free()
    return got


@pytest.mark.parametrize("size", [(1, 1), (37, 3), (1024, 512), (1500, 901)])
@pytest.mark.parametrize("pinned", [(0, 1, 2, 3), (0,), (1, 3), (2,)])
@pytest.mark.parametrize("wide", [False, True])
def test_pinned_arrays(ctx, setup, size, pinned, wide):  # noqa: F811
    sc, srv = setup
    _same(_take(ctx, srv, sc, size, pinned, wide), _plain(ctx, sc, *size))


def test_threads_take_into_pinned_and_ordinary_memory(ctx, setup):  # noqa: F811
    sc, srv = setup
    jobs = [((1500, 901), (0, 1, 2, 3)), ((1201, 700), ()), ((1024, 512), (0, 2))]
    refs = [_plain(ctx, sc, *size) for size, _ in jobs]
    errors = []

    def run(k):
        try:
            for _ in range(4):
                _same(_take(ctx, srv, sc, *jobs[k], wide=False), refs[k])
        except BaseException as e:  # surfaced after the join
            errors.append(e)

    threads = [threading.Thread(target=run, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
