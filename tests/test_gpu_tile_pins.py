"""VX_TILE_ROWS and the choices it pins: what a run reports of its fused stage's
strips pins another run to the same choice, for every form."""
import math

import pytest

import veritas_amd as va

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("codes", [[16] * 6, [4112] + [9] * 5, [8200] * 6, [8204, 16, 8196, 4104, 8200, 8]])
def test_the_reported_choice_pins_it(monkeypatch, codes):
    monkeypatch.setenv("VX_TILE_ROWS", ",".join(map(str, codes)))
    g = va.Run(va.two_stream(nx=64, np=132, length=4 * math.pi, amplitude=0.05))
    assert g.tile_code() == [0] * 6
    g.advance(g.calc_dt(0.4))
    assert g.tile_code() == codes
    assert [c % 4096 for c in g.tile_code()] == g.tile_rows()
    g.close()


def test_a_timed_choice_pins_another_run(monkeypatch):
    p = va.two_stream(nx=74, np=134, length=4 * math.pi, amplitude=0.05)
    g = va.Run(p)
    g.advance(g.calc_dt(0.4))
    codes = g.tile_code()
    assert min(codes) > 0
    monkeypatch.setenv("VX_TILE_ROWS", ",".join(map(str, codes)))
    h = va.Run(p)
    h.advance(h.calc_dt(0.4))
    assert h.tile_code() == codes
    for r in (g, h):
        r.close()
