"""Copies between the device and pageable host memory through the pinned
buffers (2 MiB each): sizes of one value, of a partial and of many chunks, byte
counts that are no whole doubles, patch rows that fill, cross and exceed a
buffer.  Every byte comes back, and bytes beside the copied range stay."""
import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import kernels

pytestmark = pytest.mark.gpu

P = ctypes.c_void_p


class Patch(ctypes.Structure):  # vx_patch
    _fields_ = ([(n, ctypes.c_int32) for n in ("n_x", "n_p", "x_pos", "p_pos", "rtb", "pitch", "l", "r", "d", "u")]
                + [(n, ctypes.c_double) for n in ("dx", "dp", "pmin", "q", "m", "dx_inv", "dp_inv", "cc", "mc2inv")]
                + [("planes", P * 26)])


@pytest.fixture(scope="module")
def lib():
    L = kernels()
    L.vx_patch_upload.argtypes = L.vx_patch_download.argtypes = [P, ctypes.POINTER(Patch), ctypes.c_int, ctypes.c_int, P]
    ctx = P()
    assert L.vx_ctx_create(0, ctypes.byref(ctx)) == 0
    yield L, ctx
    L.vx_ctx_destroy(ctx)


@pytest.mark.parametrize("nbytes", [0, 8, 13, 4096, 8192, 8200, 2 << 20, (2 << 20) + 8, (4 << 20) + 24, 11_000_008, 5_000_001])
def test_contiguous_copies(lib, nbytes):
    L, ctx = lib
    rng = np.random.default_rng(nbytes)
    a = rng.integers(0, 256, nbytes + 64, dtype=np.uint8)
    d = P()
    assert L.vx_malloc(ctx, nbytes + 64, ctypes.byref(d)) == 0
    assert L.vx_memcpy_h2d(ctx, d, a.ctypes.data, nbytes + 64) == 0
    b = rng.integers(0, 256, nbytes, dtype=np.uint8)
    assert L.vx_memcpy_h2d(ctx, d.value + 16, b.ctypes.data, nbytes) == 0
    got = np.full(nbytes + 128, 7, dtype=np.uint8)
    assert L.vx_memcpy_d2h(ctx, got.ctypes.data, d, nbytes + 64) == 0
    want = a.copy()
    want[16:16 + nbytes] = b
    assert np.array_equal(got[:nbytes + 64], want) and (got[nbytes + 64:] == 7).all()
    L.vx_free(ctx, d)


@pytest.mark.parametrize("nx,np_", [(1, 1), (5, 9), (700, 1000), (3, 262140), (3, 262144), (2, 262146), (40, 130000)])
@pytest.mark.parametrize("g", [0, 1, 2])
def test_patch_copies(lib, nx, np_, g):
    L, ctx = lib
    pitch = (np_ + 11) // 8 * 8
    n = (nx + 4) * pitch
    d = P()
    assert L.vx_malloc(ctx, 8 * n, ctypes.byref(d)) == 0
    full = np.random.default_rng(nx + np_).standard_normal((nx + 4, pitch))
    assert L.vx_memcpy_h2d(ctx, d, full.ctypes.data, 8 * n) == 0
    p = Patch(n_x=nx, n_p=np_, rtb=1, pitch=pitch)
    p.planes[0] = d.value
    inner = np.random.default_rng(1).standard_normal((nx + 2 * g, np_ + 2 * g))
    assert L.vx_patch_upload(ctx, ctypes.byref(p), 0, g, inner.ctypes.data) == 0
    full[2 - g:2 + nx + g, 2 - g:2 + np_ + g] = inner
    got = np.empty_like(full)
    assert L.vx_memcpy_d2h(ctx, got.ctypes.data, d, 8 * n) == 0
    assert np.array_equal(got, full)
    back = np.empty_like(inner)
    assert L.vx_patch_download(ctx, ctypes.byref(p), 0, g, back.ctypes.data) == 0
    assert np.array_equal(back, inner)
    L.vx_free(ctx, d)
