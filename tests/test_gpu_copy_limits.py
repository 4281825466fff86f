"""Copies that reach outside what they may touch: HIP's own copies refuse a null
address and a count past the allocation, and so do the copies through the
pinned buffers, with VX_EHIP and nothing written.  A shape without cells copies
nothing.  Sizes around those where the way of a copy changes, from pageable and from
pinned memory, keep every byte."""
import ctypes

import numpy as np
import pytest
import torch

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


@pytest.mark.parametrize("nbytes", [8, 1000, 16384, 16392, 24576, (2 << 20) - 8, 2 << 20, (2 << 20) + 8, 9_000_016])
@pytest.mark.parametrize("pinned", [False, True])
def test_copies_around_the_sizes_where_the_way_changes(lib, nbytes, pinned):
    L, ctx = lib
    d = P()
    assert L.vx_malloc(ctx, nbytes + 64, ctypes.byref(d)) == 0
    rng = np.random.default_rng(nbytes)
    up, down = (torch.empty(nbytes + 64, dtype=torch.uint8, pin_memory=pinned) for _ in range(2))
    a, b = up.numpy(), down.numpy()
    a[:] = rng.integers(0, 256, a.size)
    assert L.vx_memcpy_h2d(ctx, d, a.ctypes.data, a.size) == 0
    a[8:8 + nbytes] = rng.integers(0, 256, nbytes)
    assert L.vx_memcpy_h2d(ctx, d.value + 8, a.ctypes.data + 8, nbytes) == 0
    b[:] = 7
    assert L.vx_memcpy_d2h(ctx, b.ctypes.data + 16, d.value + 16, nbytes) == 0
    assert np.array_equal(b[16:16 + nbytes], a[16:16 + nbytes]) and (b[:16] == 7).all() and (b[16 + nbytes:] == 7).all()
    nx, np_ = 5, nbytes // 8 // 5  # the same memory as the rows of a patch
    if np_ > 12:
        p = Patch(n_x=nx - 4, n_p=np_ // 8 * 8 - 4, rtb=1, pitch=np_ // 8 * 8)
        p.planes[0] = d.value
        n = nx * p.pitch * 8
        assert L.vx_patch_download(ctx, ctypes.byref(p), 0, 2, b.ctypes.data + 16) == 0
        assert np.array_equal(b[16:16 + n], a[:n])
        a[:n] = rng.integers(0, 256, n)
        assert L.vx_patch_upload(ctx, ctypes.byref(p), 0, 2, a.ctypes.data) == 0
        assert L.vx_memcpy_d2h(ctx, b.ctypes.data, d, n) == 0 and np.array_equal(b[:n], a[:n])
    L.vx_free(ctx, d)
