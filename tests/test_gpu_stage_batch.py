"""The shared stage launch (vx_fct_stage_fused_batch) against each item's own call,
bit for bit, over the six stages: at the total size where the launch goes from a
wavefront per row to strips and one row past it, in FP64, in mixed precision and
with both, ragged patches with and without a pulse and one of 8 x 8 cells among
them; and pinned through VX_TILE_ROWS in every form."""
import ctypes

import numpy as np
import pytest
import torch

from test_gpu_moments import Fields
from test_gpu_staged_copies import P, Patch
from test_zz_no_alloc import kernels

pytestmark = pytest.mark.gpu

D = ctypes.c_double
ROWS_PER_SIMD = 20  # up to which a shared launch takes the row form


class StageItem(ctypes.Structure):  # vx_stage_item
    _fields_ = [("p", Patch), ("fl", Fields), ("fin", P), ("fout", P), ("dt", D), ("f_scale", D)]


def columns(np_):
    return (np_ + 57) // 58


def shapes(total):
    """Patches whose rows times p-columns of wavefronts add up to `total`."""
    s = [(301, 333), (8, 8), (97, 58), (640, 514), (33, 1000), (1200, 130)]
    rest = total - sum(nx * columns(np_) for nx, np_ in s)
    s += [(rest // 2 // columns(300), 300)]
    rest = total - sum(nx * columns(np_) for nx, np_ in s)
    return s + [(rest, 57)]  # one p-column


class Items:
    """Two copies of the items' planes: `one` for their own calls, `all_` for the
    shared ones."""

    def __init__(self, L, shapes, mixed):
        self.L, self.mixed, self.keep = L, mixed, []
        self.ctx = P()
        assert L.vx_ctx_create(0, ctypes.byref(self.ctx)) == 0
        rng = np.random.default_rng(11)
        self.items = []
        for k, (nx, np_) in enumerate(shapes):
            pitch = (np_ + 11) // 8 * 8
            f = np.zeros((nx + 4, pitch))
            u = (np.arange(np_) + 0.5) / np_ - 0.5
            f[2:2 + nx, 2:2 + np_] = np.exp(-80 * u * u) * (1 + 0.5 * rng.random((nx, 1))) + 1e-9 * rng.random((nx, np_))
            x = np.arange(nx + 1) / nx
            a2 = [0.3 * np.sin(9 * x + s) ** 2 if k % 2 else np.zeros(nx + 1) for s in range(6)]
            E = [np.sin(7 * x[:-1] + 0.1 * s) for s in range(6)]
            fl = []
            for s in range(6):
                q = Fields(n_f=nx, n_prepad=2, n_e=nx + 4, E=self.put(E[s]), a2=self.put(a2[s]))
                q.E0, q.a20 = (q.E, q.a2) if s == 0 else (fl[0].E, fl[0].a2)
                fl.append(q)
            both = []
            for _ in range(2):
                p = Patch(n_x=nx, n_p=np_, rtb=1, pitch=pitch, l=1, r=1, d=1, u=1, dx=1.0, dp=1.0 / np_, pmin=-0.5,
                          q=-1.0, m=1.0, dx_inv=1.0, dp_inv=float(np_), cc=1.0, mc2inv=0.5)
                p.planes[:] = [self.put(f)] + [self.put(0 * f) for _ in range(14)] + [None] * 11
                both.append(p)
            self.items.append((nx, np_, pitch, fl, both, 0.05 / np_, 1.5 if mixed(k) else 0.0))

    def put(self, a):
        t = torch.from_numpy(np.ascontiguousarray(a)).cuda()
        self.keep.append(t)
        return t.data_ptr()

    def run(self):
        """The six stages item by item and shared; the shared launches' codes."""
        L, codes = self.L, []
        torch.cuda.synchronize()
        for s in range(6):
            src = 0 if s == 0 else 1 + (s + 1) % 2
            arr = (StageItem * len(self.items))()
            for it, (nx, np_, pitch, fl, both, dt, scale) in zip(arr, self.items):
                p = both[0]
                args = [self.ctx, ctypes.byref(p), s, dt, ctypes.byref(fl[s]), p.planes[src], p.planes[1 + s % 2]]
                rc = L.vx_fct_stage_fused_mp(*args, scale) if scale else L.vx_fct_stage_fused(*args)
                assert rc == 0, L.vx_last_error(self.ctx)
                p = both[1]
                it.p, it.fl, it.dt, it.f_scale = p, fl[s], dt, scale
                it.fin, it.fout = p.planes[src], p.planes[1 + s % 2]
            assert L.vx_fct_stage_fused_batch(self.ctx, arr, len(arr), s) == 0, L.vx_last_error(self.ctx)
            codes.append([L.vx_stage_tile_code(self.ctx, 0, 0, s, m) for m in (0, 1)])
            for nx, np_, pitch, _, both, _, _ in self.items:
                n = (nx + 4) * pitch
                got = [np.empty(n) for _ in range(2)]
                for plane in [1 + s % 2] + ([3 + s, 9 + s] if s < 5 else []):
                    for g, p in zip(got, both):
                        assert L.vx_memcpy_d2h(self.ctx, g.ctypes.data, p.planes[plane], 8 * n) == 0
                    assert np.array_equal(*got), (s, nx, np_, plane)
                    assert np.isfinite(got[0]).all() and np.abs(got[0]).max() > 0
        return codes

    def free(self):
        self.L.vx_ctx_destroy(self.ctx)


@pytest.fixture(scope="module")
def lib():
    L = kernels()
    pp, pf = ctypes.POINTER(Patch), ctypes.POINTER(Fields)
    L.vx_fct_stage_fused.argtypes = [P, pp, ctypes.c_int, D, pf, P, P]
    L.vx_fct_stage_fused_mp.argtypes = L.vx_fct_stage_fused.argtypes + [D]
    L.vx_fct_stage_fused_batch.argtypes = [P, ctypes.POINTER(StageItem), ctypes.c_int, ctypes.c_int]
    L.vx_stage_tile_code.argtypes = [P, ctypes.c_int32, ctypes.c_int32, ctypes.c_int, ctypes.c_int]
    return L


def border():
    return ROWS_PER_SIMD * 4 * torch.cuda.get_device_properties(0).multi_processor_count


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("past", [0, 1])
def test_shared_launch_on_either_side_of_the_rule(lib, mixed, past):
    c = Items(lib, shapes(border() + past), lambda k: mixed)
    codes = c.run()
    for code in (q[mixed] for q in codes):
        assert code < 4096 if past else code == 8192 + 12
    assert all(q[not mixed] == 0 for q in codes)
    c.free()


def test_shared_launch_of_both_precisions(lib):
    """The FP64 items in strips, the mixed ones as rows, and the other way round."""
    big, small = shapes(border() + 1), [(301, 333), (8, 8), (97, 58)]
    for swap in (False, True):
        c = Items(lib, small + big, lambda k: (k < len(small)) != swap)
        for fp64, mixed in c.run():
            assert (mixed if swap else fp64) < 4096 and (fp64 if swap else mixed) == 8192 + 12
        c.free()


@pytest.mark.parametrize("code", [1, 9, 64, 4105, 8193, 8196, 8203, 8204])
def test_pinned_shared_launch(lib, code, monkeypatch):
    monkeypatch.setenv("VX_TILE_ROWS", str(code))
    c = Items(lib, [(37, 130), (8, 8), (150, 60)], lambda k: k == 2)
    want = code if code > 8192 else code % 4096
    assert c.run() == [[want, want]] * 6
    c.free()
