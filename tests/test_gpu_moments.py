"""The p-moments (k_moments) against the oracle, bit for bit: column counts that
leave a partial workgroup, p-columns that end inside, at and just past a 64-cell
chunk, tall columns (8 a workgroup from 2048 p-cells on), patches with and
without the logarithm table (above 2^20 cells), with and without nested cells
(levels 3: relativeToBottom 1, 2 and 4), behind and ahead of a pulse.  The
compensated sums agree with the ordered ones.  A table of another patch is never
taken for this one's, a recorded launch keeps its own, several patches in one launch give each one's bits, and a
patch that is the whole grid writes what the assembly would."""
import ctypes

import numpy as np
import pytest

import veritas_amd as va
from _amr_cases import two_slab_laser
from _oracle import OracleRun
from test_gpu_parity import assert_same
from test_gpu_staged_copies import Patch
from test_zz_no_alloc import kernels

pytestmark = pytest.mark.gpu

SHAPES = [(1, 8, 8), (1, 10, 62), (1, 34, 64), (1, 30, 66), (1, 12, 128), (1, 1026, 1022), (1, 1026, 1030),
          (1, 10, 2046), (1, 10, 2048), (1, 14, 2050), (1, 522, 2050),
          (3, 128, 64), (3, 126, 66), (3, 1026, 514)]


@pytest.mark.parametrize("levels,nx,np_", SHAPES)
def test_moments_match_the_oracle(levels, nx, np_):
    p = two_slab_laser(levels=levels, nx=nx, np=np_)
    g, o = va.Run(p, fused=False), OracleRun(p)
    dt = o.calc_dt(0.4)
    g.advance(dt, 2)  # the pulse has entered the first columns
    o.advance(dt, 2)
    assert levels == 3 or np.any(o.get("a2") != 0)
    g.stage_moments()
    q, j = o.moments()
    q0, j0 = g.get("charge"), g.get("J")
    assert_same("charge", q0, q)
    assert_same("J", j0, j)
    # a compensated sum is exact to an ulp of itself, an ordered one of n terms of
    # one sign to n 2^-53; a column has at most 4 np_ cells
    g.set_mixed(True)
    g.stage_moments()
    tol = (4 * np_ + 8) * 2.0**-53
    for a, b in ((g.get("charge"), q0), (g.get("J"), j0)):
        assert np.abs(a - b).max() <= tol * np.abs(b).max()
    g.close()
    o.close()


class Fields(ctypes.Structure):  # vx_fields
    _fields_ = ([(n, ctypes.c_int32) for n in ("n_f", "n_prepad", "n_e", "pad")]
                + [(n, ctypes.c_void_p) for n in ("E", "a2", "Ay1", "Az1", "E0", "a20")])


class Case:
    """Patches of the given (n_x, n_p, rtb, nested) in one context, with an A^2
    that is 0, uniform or varies."""

    def __init__(self, shapes, a):
        L = self.L = kernels()
        pp, pf = ctypes.POINTER(Patch), ctypes.POINTER(Fields)
        L.vx_moments_patch.argtypes = L.vx_moments_patch_compensated.argtypes = [ctypes.c_void_p, pp, pf]
        L.vx_moments_patches.argtypes = [ctypes.c_void_p, pp, ctypes.c_int32, pf, ctypes.c_int]
        self.ctx, self.bufs = ctypes.c_void_p(), []
        assert L.vx_ctx_create(0, ctypes.byref(self.ctx)) == 0
        rng = np.random.default_rng(3)
        n_f = max(nx * rtb for nx, _, rtb, _ in shapes)
        self.p, self.out = (Patch * len(shapes))(), []
        for k, (nx, np_, rtb, nested) in enumerate(shapes):
            pitch = (np_ + 11) // 8 * 8
            f = rng.uniform(1.0, 2.0, (nx + 4, pitch))
            mask = (rng.random((nx + 4, pitch)) < 0.4).astype(np.uint8)
            planes = [self.put(f)] * 3 + [None] * 20 + [self.put(mask) if nested else None]
            self.out.append([self.put(np.zeros(nx * rtb)) for _ in range(2)])
            self.p[k] = Patch(n_x=nx, n_p=np_, rtb=rtb, pitch=pitch, l=1, r=1, d=1, u=1, dx=1.0, dp=0.004,
                                  pmin=-0.002 * np_, q=-1.0, m=1.0, dx_inv=1.0, dp_inv=250.0, cc=9e16, mc2inv=0.5)
            self.p[k].planes[:] = [None if q is None else q.value for q in planes + self.out[-1]]
        self.fl = Fields(n_f=n_f, n_prepad=2, n_e=n_f + 4)
        x = np.arange(n_f + 4)
        A = {"zero": 0.0 * x, "uniform": 0.6 + 0.0 * x, "pulse": np.maximum(0.0, np.sin(x / 40.0))}[a]
        for name in ("E", "a2", "Ay1", "Az1", "E0", "a20"):
            setattr(self.fl, name, self.put(A).value)

    def put(self, a):
        d = ctypes.c_void_p()
        a = np.ascontiguousarray(a)
        assert self.L.vx_malloc(self.ctx, a.nbytes, ctypes.byref(d)) == 0
        assert self.L.vx_memcpy_h2d(self.ctx, d, a.ctypes.data, a.nbytes) == 0
        self.bufs.append(d)
        return d

    def get(self, k):
        """The charge and current of patch k, which are then cleared."""
        got = []
        for d in self.out[k]:
            a = np.empty(self.p[k].n_x * self.p[k].rtb)
            assert self.L.vx_memcpy_d2h(self.ctx, a.ctypes.data, d, a.nbytes) == 0
            z = np.zeros_like(a)
            assert self.L.vx_memcpy_h2d(self.ctx, d, z.ctypes.data, z.nbytes) == 0
            got.append(a)
        return got

    def one(self, k, comp=False):
        f = self.L.vx_moments_patch_compensated if comp else self.L.vx_moments_patch
        assert f(self.ctx, ctypes.byref(self.p[k]), ctypes.byref(self.fl)) == 0, self.L.vx_last_error(self.ctx)
        return self.get(k)

    def free(self):
        for d in self.bufs:
            self.L.vx_free(self.ctx, d)
        self.L.vx_ctx_destroy(self.ctx)


@pytest.mark.parametrize("comp", [False, True])
@pytest.mark.parametrize("shape", [(37, 70, 1, False), (20, 2050, 1, False), (9, 130, 4, True), (16, 64, 2, False)])
def test_whole_patch_writes_the_assembled_moments(shape, comp):
    """0.0 + the patch's own moments, as the assembly forms them, in charge, J and the
    species' charge; columns without particles give +0.0."""
    c = Case([shape], "pulse")
    L, n = c.L, shape[0] * shape[2]
    L.vx_moments_whole.argtypes = [ctypes.c_void_p, ctypes.POINTER(Patch), ctypes.POINTER(Fields), ctypes.c_int] + \
        [ctypes.c_void_p] * 3
    c.p[0].planes[1] = c.put(np.where(np.arange(shape[0] + 4)[:, None] < 8, 0.0, 1.5)
                             * np.ones((1, c.p[0].pitch))).value
    q, j = c.one(0, comp)
    assert np.signbit(q[0]) and q[0] == 0.0
    out = [c.put(np.full(n, 7.0)) for _ in range(3)]
    assert L.vx_moments_whole(c.ctx, ctypes.byref(c.p[0]), ctypes.byref(c.fl), comp, *out) == 0
    for d, want in zip(out, (q, j, q)):
        a = np.empty(n)
        assert L.vx_memcpy_d2h(c.ctx, a.ctypes.data, d, a.nbytes) == 0
        assert np.array_equal(a.view(np.int64), (0.0 + want).view(np.int64))
    c.p[0].x_pos = 1
    assert L.vx_moments_whole(c.ctx, ctypes.byref(c.p[0]), ctypes.byref(c.fl), comp, *out) != 0
    c.free()


def test_patches_of_different_heights_in_turn():
    """Two patches above the table's size with one A^2, the second short enough
    that its tables end inside the first one's entries: the first patch's moments
    are the same before and after the second's."""
    c = Case([(960, 1100, 1, False), (3520, 300, 1, False)], "uniform")
    first, _, again = c.one(0), c.one(1), c.one(0)
    assert np.abs(first).min() > 0 and np.array_equal(first, again)
    c.free()


@pytest.mark.parametrize("a", ["zero", "uniform", "pulse"])
@pytest.mark.parametrize("comp", [False, True])
def test_patches_together_match_each_alone(a, comp):
    """More patches than one launch holds, of every relativeToBottom, with and
    without nested cells, below and above the table's size (alone they read it,
    together they form their logarithms) and one that keeps its own launch: the
    same bits as each alone."""
    c = Case([(2050, 1030, 1, False), (1030, 1022, 1, False), (1030, 1022, 2, True), (2200, 500, 4, True),
              (1030, 1026, 4, False), (7, 9, 1, False), (33, 64, 2, False), (5, 130, 4, True), (64, 65, 1, True),
              (1, 8, 4, False), (130, 100, 2, True), (18, 192, 1, False), (40, 66, 4, False), (9, 127, 2, True),
              (3, 1, 1, False)], a)
    n = len(c.p)
    alone = [c.one(k, comp) for k in range(n)]
    for m in (n, 12, 13, 1):
        assert c.L.vx_moments_patches(c.ctx, c.p, m, ctypes.byref(c.fl), comp) == 0, c.L.vx_last_error(c.ctx)
        for k in range(n):
            for x, y in zip(c.get(k), alone[k]):
                assert np.array_equal(x, y if k < m else 0.0 * y), (k, m)
    assert all(np.abs(y).max() > 0 for r in alone for y in r)
    c.free()


def test_a_recorded_launch_outlives_its_logarithm_table():
    """A graph recorded with one table, replayed after a taller patch of the same
    context needed a larger one, between eager calls of both."""
    c = Case([(1030, 1030, 1, False), (300, 4100, 1, False), (200, 8200, 1, False)], "uniform")
    L = c.L
    L.vx_graph_begin.argtypes, L.vx_graph_destroy.argtypes = [ctypes.c_void_p], [ctypes.c_void_p]
    L.vx_graph_end.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p)]
    L.vx_graph_launch.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    want, g = c.one(0), ctypes.c_void_p()
    assert L.vx_graph_begin(c.ctx) == 0
    assert L.vx_moments_patch(c.ctx, ctypes.byref(c.p[0]), ctypes.byref(c.fl)) == 0
    assert L.vx_graph_end(c.ctx, ctypes.byref(g)) == 0
    tall = {}
    for k in (1, 1, 2, 1, 2, 0):
        got = c.one(k)
        assert np.array_equal(got, tall.setdefault(k, got))
        assert L.vx_graph_launch(c.ctx, g) == 0
        assert np.array_equal(c.get(0), want)
        # memory taken now, which a freed table's place would serve, keeps its values
        q = np.full(4096, 3.0)
        d, back = c.put(q), np.empty(4096)
        assert L.vx_graph_launch(c.ctx, g) == 0
        assert np.array_equal(c.get(0), want)
        assert L.vx_memcpy_d2h(c.ctx, back.ctypes.data, d, back.nbytes) == 0
        assert np.array_equal(back, q)
    assert np.array_equal(tall[0], want) and np.abs(want).min() > 0
    L.vx_graph_destroy(g)
    c.free()


@pytest.mark.parametrize("comp", [False, True])
@pytest.mark.parametrize("shape", [(37, 70, 1, False), (20, 2050, 1, False), (9, 130, 4, True)])
def test_whole_patch_keeps_its_own_moments(shape, comp):
    """The patch's chargeR and currentR after the call that assembles them: those of
    the patch's own call; a patch without them is accepted."""
    c = Case([shape], "pulse")
    c.L.vx_moments_whole.argtypes = [ctypes.c_void_p, ctypes.POINTER(Patch), ctypes.POINTER(Fields), ctypes.c_int] + \
        [ctypes.c_void_p] * 3
    want, out = c.one(0, comp), [c.put(np.zeros(shape[0] * shape[2])) for _ in range(3)]
    args = c.ctx, ctypes.byref(c.p[0]), ctypes.byref(c.fl), comp, *out
    assert c.L.vx_moments_whole(*args) == 0
    for got, ref in zip(c.get(0), want):
        assert np.array_equal(got, ref) and np.abs(ref).max() > 0
    c.p[0].planes[24] = c.p[0].planes[25] = None
    assert c.L.vx_moments_whole(*args) == 0
    c.free()


@pytest.mark.parametrize("a", ["zero", "uniform", "pulse"])
@pytest.mark.parametrize("comp", [False, True])
def test_tall_patches_around_the_rules(a, comp):
    """Heights on either side of those from which a small rtb 1 patch has a table, alone
    (with it) and in one launch with another (without); full launches of tall columns
    (8 a workgroup) with a ragged last workgroup, against a part of their columns."""
    tall = [(10, 1022, 1, False), (9, 1026, 1, False), (6, 1088, 2, True), (10, 1536, 1, False), (11, 1538, 1, False),
            (7, 1602, 4, False), (5, 1600, 1, True), (70, 2050, 1, False)]
    c = Case(tall + [(2050, 2050, 1, False), (1030, 2050, 1, False)], a)
    n = len(tall)
    alone = [c.one(k, comp) for k in range(n)]
    assert c.L.vx_moments_patches(c.ctx, c.p, n, ctypes.byref(c.fl), comp) == 0
    for k in range(n):
        for x, y in zip(c.get(k), alone[k]):
            assert np.array_equal(x, y) and np.abs(y).max() > 0, k
    full = c.one(n, comp)
    c.p[n + 1].planes[1] = c.p[n].planes[1]  # the first columns of the same f
    for x, y in zip(c.one(n + 1, comp), full):
        assert np.array_equal(x, y[:1030]) and np.abs(y).min() > 0
    c.free()


def test_a_tall_patch_recorded_before_there_is_a_table():
    c = Case([(10, 1602, 1, False)], "uniform")
    L, g = c.L, ctypes.c_void_p()
    L.vx_graph_begin.argtypes, L.vx_graph_destroy.argtypes = [ctypes.c_void_p], [ctypes.c_void_p]
    L.vx_graph_end.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p)]
    L.vx_graph_launch.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    assert L.vx_graph_begin(c.ctx) == 0
    assert L.vx_moments_patch(c.ctx, ctypes.byref(c.p[0]), ctypes.byref(c.fl)) == 0
    assert L.vx_graph_end(c.ctx, ctypes.byref(g)) == 0
    want = c.one(0)
    for _ in range(3):
        assert L.vx_graph_launch(c.ctx, g) == 0
        for x, y in zip(c.get(0), want):
            assert np.array_equal(x, y) and np.abs(y).min() > 0
        c.one(0)
    L.vx_graph_destroy(g)
    c.free()
