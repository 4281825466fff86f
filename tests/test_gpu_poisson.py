"""vx_poisson at the edges of its forms (wavefronts, entries a thread, sub-chunks
of 64, chunks of 192 and 512, the solvers' borders at 4096 and 36864), through
the C ABI, against the oracle's solve of the same right-hand side: both converge
to the correctly rounded solution (a near-tie may differ by 1 ulp), E and Ex0
follow from phi.  Smooth, random and zero charges; a second call repeats the
first's bits."""
import ctypes

import numpy as np
import pytest

import veritas_amd as va
from _oracle import OracleRun
from test_gpu_parity import assert_ulp
from test_zz_no_alloc import State, kernels

pytestmark = pytest.mark.gpu

SIZES = [8, 10, 16, 34, 64, 66, 128, 130, 256, 258, 512, 514, 1024, 1026, 2048, 2050, 4094, 4096,
         4098, 4114, 4160, 4162, 4224, 4226, 4606, 4608, 4610, 4628, 8190, 8192, 10000, 20002, 36864, 36866,
         40000, 65536, 70000]
EPS0_INV = 1.1294e+11


@pytest.fixture(scope="module")
def lib():
    L = kernels()
    ctx = ctypes.c_void_p()
    assert L.vx_ctx_create(0, ctypes.byref(ctx)) == 0
    yield L, ctx
    L.vx_ctx_destroy(ctx)


@pytest.mark.parametrize("n_f", SIZES)
def test_poisson_matches_the_oracle(lib, n_f):
    L, ctx = lib
    print(f"case: n_f = {n_f}", flush=True)
    o = OracleRun(va.landau(nx=n_f, np=8))
    rng = np.random.default_rng(n_f)
    x = np.arange(n_f) / n_f
    for kind in ("smooth", "random", "zero"):
        ch = {"smooth": 1e3 * np.sin(2 * np.pi * (3 * x + 0.1)) - 1e6,
              "random": rng.normal(0.0, 1e5, n_f), "zero": np.full(n_f, 7.0)}[kind]
        ne = {"smooth": np.full(n_f, 1e6), "random": -np.roll(ch, 3) * 0.999, "zero": np.full(n_f, -7.0)}[kind]
        s = State(L, ctx, n_f, ch, ne, 0.25, work=True)
        b = EPS0_INV * (ch + ne)
        b = b * s.fs.dx2
        ref = o.poisson(b)
        ex0 = 0.25
        for call in range(2):
            assert L.vx_poisson(ctx, ctypes.byref(s.fs)) == 0, L.vx_last_error(ctx)
            phi = s.get("phi", n_f)
            assert np.abs(ref).max() > 0 or kind == "zero"
            assert_ulp(f"{kind} phi", phi, ref)
            fc = s.fs.field_coef
            d = 8 * (np.roll(phi, -1) - np.roll(phi, 1)) - np.roll(phi, -2) + np.roll(phi, 2)
            e = -fc * d + ex0
            ex0 = ex0 + -(e[-1] + e[0]) * 0.5
            assert s.get("Ex0", 1)[0] == ex0
            assert np.array_equal(s.get("E", n_f), -fc * d + ex0)
        s.free()


@pytest.mark.parametrize("n_f", [131070, 131072, 131074, 200002, 263170])
def test_poisson_of_many_cells_matches_the_oracle(lib, n_f):
    """Either side of the border at 131072 cells, where each compute unit has a chunk."""
    test_poisson_matches_the_oracle(lib, n_f)
