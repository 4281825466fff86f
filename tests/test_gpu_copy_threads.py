"""Threads that copy to and from the device on one context at once, each its own
arrays: every thread gets its own values, whole."""
import ctypes
import threading

import numpy as np
import pytest

from test_gpu_staged_copies import P, Patch, lib

pytestmark = pytest.mark.gpu


def together(n, work):
    """work(k) in n threads; the first exception is raised here."""
    errors, start = [], threading.Barrier(n)

    def body(k):
        try:
            start.wait()
            work(k)
        except BaseException as e:  # noqa: BLE001 (reported below)
            errors.append(e)
    t = [threading.Thread(target=body, args=(k,)) for k in range(n)]
    for q in t:
        q.start()
    for q in t:
        q.join()
    if errors:
        raise errors[0]


@pytest.mark.parametrize("nx,np_", [(3, 5), (64, 256), (700, 1000)])
def test_threads_copy_patches_and_arrays_of_one_context(lib, nx, np_):
    L, ctx = lib
    pitch = (np_ + 11) // 8 * 8
    n = (nx + 4) * pitch
    dev = [P() for _ in range(4)]
    for d in dev:
        assert L.vx_malloc(ctx, 8 * n, ctypes.byref(d)) == 0

    def work(k):
        rng = np.random.default_rng(k)
        p = Patch(n_x=nx, n_p=np_, rtb=1, pitch=pitch)
        p.planes[0] = dev[k].value
        got, back = np.empty((nx + 4, pitch)), np.empty((nx, np_))
        for _ in range(16):
            f, inner = rng.standard_normal((nx + 4, pitch)), rng.standard_normal((nx, np_))
            assert L.vx_memcpy_h2d(ctx, dev[k], f.ctypes.data, 8 * n) == 0
            assert L.vx_patch_upload(ctx, ctypes.byref(p), 0, 0, inner.ctypes.data) == 0
            f[2:2 + nx, 2:2 + np_] = inner
            assert L.vx_memcpy_d2h(ctx, got.ctypes.data, dev[k], 8 * n) == 0
            assert np.array_equal(got, f), k
            assert L.vx_patch_download(ctx, ctypes.byref(p), 0, 0, back.ctypes.data) == 0
            assert np.array_equal(back, inner), k
    together(4, work)
    for d in dev:
        L.vx_free(ctx, d)
