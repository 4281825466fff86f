"""Copies that reach outside what they may touch: HIP's own copies refuse a null
address and a count past the allocation, and so do the copies through the
pinned buffers, with VX_EHIP and nothing written.  A shape without cells copies
nothing."""
import ctypes

import numpy as np
import pytest

from test_gpu_staged_copies import P, Patch, lib

pytestmark = pytest.mark.gpu

VX_EHIP = -2


@pytest.fixture
def block(lib):
    """Two allocations of 4608 bytes (a page and an eighth) holding 0, 1, 2, ..."""
    L, ctx = lib
    a = np.arange(576.0)
    d = [P(), P()]
    for q in d:
        assert L.vx_malloc(ctx, 4608, ctypes.byref(q)) == 0
        assert L.vx_memcpy_h2d(ctx, q, a.ctypes.data, 4608) == 0
    yield d[0].value
    for q in d:
        got = np.empty(576)
        assert L.vx_memcpy_d2h(ctx, got.ctypes.data, q, 4608) == 0
        assert np.array_equal(got, a)
        L.vx_free(ctx, q)


@pytest.mark.parametrize("offset,nbytes", [(None, 8), (0, 4616), (8, 4608), (4600, 16)])
def test_contiguous_copies_stay_inside_the_allocation(lib, block, offset, nbytes):
    L, ctx = lib
    h = np.full(1024, -1.0)
    at = None if offset is None else block + offset
    assert L.vx_memcpy_h2d(ctx, at, h.ctypes.data, nbytes) == VX_EHIP and L.vx_last_error(ctx)
    assert L.vx_memcpy_d2h(ctx, h.ctypes.data, at, nbytes) == VX_EHIP
    assert (h == -1.0).all()
    assert L.vx_memcpy_h2d(ctx, block, None, 8) == VX_EHIP
    assert L.vx_memcpy_d2h(ctx, None, block, 8) == VX_EHIP


@pytest.mark.parametrize("nx,np_,pitch", [(9, 44, 48), (8, 45, 40), (72, 4, 8)])
def test_patch_copies_stay_inside_the_allocation(lib, block, nx, np_, pitch):
    """A plane of more rows than the allocation's, and rows longer than the pitch."""
    L, ctx = lib
    p = Patch(n_x=nx, n_p=np_, rtb=1, pitch=pitch)
    p.planes[0] = block
    h = np.full((nx + 4) * (np_ + 4), -1.0)
    assert L.vx_patch_upload(ctx, ctypes.byref(p), 0, 2, h.ctypes.data) == VX_EHIP
    assert L.vx_patch_download(ctx, ctypes.byref(p), 0, 2, h.ctypes.data) == VX_EHIP
    assert (h == -1.0).all()


@pytest.mark.parametrize("nx,np_,g", [(4, 0, 0), (0, 4, 0), (0, 0, 0), (4, -2, 1), (-4, 4, 2)])
def test_an_empty_patch_copies_nothing(lib, block, nx, np_, g):
    L, ctx = lib
    p = Patch(n_x=nx, n_p=np_, rtb=1, pitch=8)
    p.planes[0] = block
    h = np.full(64, -1.0)
    assert L.vx_patch_upload(ctx, ctypes.byref(p), 0, g, h.ctypes.data) == 0
    assert L.vx_patch_download(ctx, ctypes.byref(p), 0, g, h.ctypes.data) == 0
    assert (h == -1.0).all()
