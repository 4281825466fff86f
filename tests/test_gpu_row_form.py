"""The fused stage with one wavefront per row (k_stage_rows), pinned through
VX_TILE_ROWS (rows + 8192), against the oracle bit for bit: row counts that
divide n_x, leave a remainder or exceed it, p-columns that end inside, at and
just past a wavefront's 58 cells, with and without a pulse in A^2, values
beyond the short divisions, and the mixed-precision form against the strips."""
import math

import numpy as np
import pytest

import veritas_amd as va
from _amr_cases import two_slab_laser
from _oracle import OracleRun
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu

SHAPES = [(64, 256), (8, 8), (14, 58), (26, 60), (48, 116), (150, 132)]


def two_stream(nx, np_, **kw):
    return va.two_stream(nx=nx, np=np_, length=4 * math.pi, amplitude=0.05, **kw)


def check(p, steps=2):
    g, o = va.Run(p, fused=True), OracleRun(p)
    dt = o.calc_dt(0.4)
    g.advance(dt, steps)
    o.advance(dt, steps)
    assert_same("f1", g.get("f1"), o.get("f1"))
    assert_same("E", g.get("E"), o.get("E"))
    tiles = g.tile_rows(), g.tile_waves()
    g.close()
    o.close()
    return tiles


@pytest.mark.parametrize("rows", [4, 8, 12, 1])
@pytest.mark.parametrize("nx,np_", SHAPES)
def test_row_form_matches_the_oracle(monkeypatch, nx, np_, rows):
    print(f"case: {nx}x{np_}, {rows} rows", flush=True)
    monkeypatch.setenv("VX_TILE_ROWS", str(8192 + rows))
    assert check(two_stream(nx, np_)) == ([rows] * 6, [4] * 6)


@pytest.mark.parametrize("rows", [4, 12])
def test_row_form_with_a_pulse_and_wide_values(monkeypatch, rows):
    monkeypatch.setenv("VX_TILE_ROWS", str(8192 + rows))
    check(two_slab_laser(levels=1), steps=12)
    check(va.landau(nx=40, np=132, n_ref=1e38))
    check(two_slab_laser(levels=1, lambda0=1e-13))


def test_row_form_between_strips(monkeypatch):
    """Stages of one step may take different forms (each is timed by itself)."""
    monkeypatch.setenv("VX_TILE_ROWS", "8204,16,8196,4104,8200,8")
    check(two_stream(150, 132))
    monkeypatch.setenv("VX_TILE_ROWS", "16,8204,4104,8196,8,8200")
    check(two_stream(150, 132))


@pytest.mark.parametrize("nx,np_", [(26, 60), (150, 132)])
def test_mixed_row_form_equals_the_mixed_strips(monkeypatch, nx, np_):
    out = []
    for rows in ("16", "8200", "8204"):
        monkeypatch.setenv("VX_TILE_ROWS", rows)
        g = va.Run(two_stream(nx, np_), mixed=True)
        dt = g.calc_dt(0.4)
        g.advance(dt, 3)
        out.append(g.get("f1"))
        g.close()
    assert np.isfinite(out[0]).all() and out[0].max() > 0
    assert_same("8 rows", out[1], out[0])
    assert_same("12 rows", out[2], out[0])
