"""The transverse fields' one-workgroup stage (up to 512 elements with the
padding) at its edges, and the two launches above it, bit for bit against the
oracle: field-only steps with the laser's drive, then full steps."""
import numpy as np
import pytest

import veritas_amd as va
from _amr_cases import two_slab_laser
from _oracle import OracleRun
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [8, 62, 250, 506, 508, 510, 512])
def test_fields_match_the_oracle(nx):
    p = two_slab_laser(levels=1, nx=nx, np=16)
    g, o = va.Run(p), OracleRun(p)
    dt = o.calc_dt(0.4)
    for step in range(2):
        g.advance_fields(dt, 7)
        o.advance_fields(dt, 7)
        assert np.any(o.get("a2") != 0)
        for w in ("By", "Bz", "Ey", "Ez", "Ay", "Az", "a2"):
            assert_same(f"{nx} {w}", g.get(w), o.get(w))
        g.advance(dt, 1)
        o.advance(dt, 1)
    assert_same(f"{nx} f1", g.get("f1"), o.get("f1"))
    for w in ("By", "Bz", "Ey", "Ez", "Ay", "Az", "a2"):
        assert_same(f"{nx} {w}", g.get(w), o.get(w))
    g.close()
    o.close()
