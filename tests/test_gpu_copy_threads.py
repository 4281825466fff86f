"""Threads that copy to and from the device on one context at once, each its own
arrays: every thread gets its own values, whole.  The CFL bound, whose maxima come
through the same pinned buffers, is the same beside copies, and it refuses field
arrays that it cannot read."""
import ctypes
import threading

import numpy as np
import pytest

from test_gpu_staged_copies import P, Patch, lib
from test_zz_no_alloc import D, FieldState, State

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


def bound(L, ctx, fs):
    """vx_cfl_bound of one electron species: (return code, bound)."""
    L.vx_cfl_bound.argtypes = [P, ctypes.POINTER(FieldState), ctypes.c_int] + [ctypes.POINTER(D)] * 4
    q, m, dp, out = D(-1.60217657e-19), D(9.10938291e-31), D(1e-24), D(-1.0)
    rc = L.vx_cfl_bound(ctx, ctypes.byref(fs), 1, ctypes.byref(q), ctypes.byref(m), ctypes.byref(dp), ctypes.byref(out))
    return rc, out.value


@pytest.fixture
def fields(lib):
    L, ctx = lib
    s = State(L, ctx, 3000, np.zeros(3000), np.zeros(3000), 0.0, work=False)
    rng = np.random.default_rng(5)
    for name, amp in (("Ay", 1e-3), ("Az", 1e-3), ("By", 1e4), ("Bz", 1e4), ("E", 1e12)):
        s.put(name, amp * rng.standard_normal(3000))
    yield s
    s.free()


def test_the_cfl_bound_beside_copies_of_the_same_context(lib, fields):
    L, ctx = lib
    rc, want = bound(L, ctx, fields.fs)
    assert rc == 0 and want > 0
    a = np.full(200_000, 1e300)  # (a bound from these values would be 0)
    d = P()
    assert L.vx_malloc(ctx, a.nbytes, ctypes.byref(d)) == 0

    def work(k):
        got = np.empty_like(a)
        for _ in range(20):
            if k == 0:
                assert bound(L, ctx, fields.fs) == (0, want)
            else:
                assert L.vx_memcpy_h2d(ctx, d, a.ctypes.data, a.nbytes) == 0
                assert L.vx_memcpy_d2h(ctx, got.ctypes.data, d, a.nbytes) == 0
                assert np.array_equal(got, a)
    together(2, work)
    L.vx_free(ctx, d)


@pytest.mark.parametrize("name", ["Ay", "Az", "By", "Bz", "E"])
def test_the_cfl_bound_refuses_arrays_that_are_not_there(lib, fields, name):
    L, ctx = lib
    was = getattr(fields.fs, name)
    setattr(fields.fs, name, None)
    assert bound(L, ctx, fields.fs) == (-2, -1.0)
    setattr(fields.fs, name, was)
    assert bound(L, ctx, fields.fs)[0] == 0
