"""A patch table whose first flux launch is a later stage's: the strip timing of
that launch changes no result.  Each stage's planes against those of a
table with pinned strips, bit for bit."""
import ctypes

import numpy as np
import pytest

from test_gpu_moments import Fields
from test_gpu_staged_copies import P, Patch
from test_zz_no_alloc import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", range(6))
@pytest.mark.parametrize("mixed", [False, True])
def test_the_table_may_start_at_any_stage(first, mixed, monkeypatch):
    L = kernels()
    pp, pf = ctypes.POINTER(Patch), ctypes.POINTER(Fields)
    L.vx_patch_table_create.argtypes = [P, pp, ctypes.c_int32, ctypes.POINTER(P)]
    L.vx_patch_table_destroy.argtypes = [P]
    for name, more in (("vx_fct_sub0_fluxes_table", []), ("vx_fct_sub0_fluxes_table_mp", [ctypes.c_double])):
        getattr(L, name).argtypes = [P, P, ctypes.c_int, ctypes.c_double, pf] + more
    ctx, bufs = P(), []
    assert L.vx_ctx_create(0, ctypes.byref(ctx)) == 0

    def put(a):
        d = P()
        assert L.vx_malloc(ctx, a.nbytes, ctypes.byref(d)) == 0
        assert L.vx_memcpy_h2d(ctx, d, a.ctypes.data, a.nbytes) == 0
        bufs.append(d)
        return d.value
    # shapes of this test's own per case, so that no choice of another table serves
    nx, np_ = 300 + first, 130 + 2 * mixed
    pitch = (np_ + 11) // 8 * 8
    rng = np.random.default_rng(first)
    f, zero = rng.uniform(1.0, 2.0, (nx + 4, pitch)), np.zeros((nx + 4, pitch))

    def case():
        p = Patch(n_x=nx, n_p=np_, rtb=1, pitch=pitch, l=1, r=1, d=1, u=1, dx=1.0, dp=0.01, pmin=-0.65, q=-1.0, m=1.0,
                  dx_inv=1.0, dp_inv=100.0, cc=1.0, mc2inv=0.5)
        p.planes[:] = [put(f)] * 3 + [put(zero) for _ in range(20)] + [None] * 3
        t = P()
        assert L.vx_patch_table_create(ctx, ctypes.byref(p), 1, ctypes.byref(t)) == 0
        return p, t
    fl = Fields(n_f=nx, n_prepad=2, n_e=nx + 4, E=put(np.sin(np.arange(nx) / 9.0)), a2=put(0.3 + 0.2 * np.sin(np.arange(nx + 1.0))))
    fl.E0, fl.a20 = fl.E, fl.a2

    def stage(table, s):
        args = (ctx, table, s, 0.01, ctypes.byref(fl))
        rc = L.vx_fct_sub0_fluxes_table_mp(*args, 1.5) if mixed else L.vx_fct_sub0_fluxes_table(*args)
        assert rc == 0, L.vx_last_error(ctx)

    n = (nx + 4) * pitch

    def planes(p):
        out = np.empty((16, n))
        for k in range(16):
            assert L.vx_memcpy_d2h(ctx, out[k].ctypes.data, p.planes[3 + k], 8 * n) == 0
        return out
    # the planes around each stage, with pinned strips (no launch is timed)
    ref, ref_table = case()
    monkeypatch.setenv("VX_AMR_POLICY", "16,16")
    want = [planes(ref)]
    for s in range(6):
        stage(ref_table, s)
        want.append(planes(ref))
    monkeypatch.delenv("VX_AMR_POLICY")
    # from stage `first` on with a table that has launched nothing yet
    new, new_table = case()
    for k in range(16):
        assert L.vx_memcpy_h2d(ctx, new.planes[3 + k], want[first][k].ctypes.data, 8 * n) == 0
    for s in range(first, 6):
        stage(new_table, s)
        assert np.array_equal(planes(new), want[s + 1]), s
    assert np.abs(want[6]).max(axis=1).min() > 0
    for t in (ref_table, new_table):
        L.vx_patch_table_destroy(t)
    for d in bufs:
        L.vx_free(ctx, d)
    L.vx_ctx_destroy(ctx)
