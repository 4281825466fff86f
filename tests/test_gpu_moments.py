"""The p-moments (k_moments) against the oracle, bit for bit: column counts that
leave a partial workgroup, p-columns that end inside, at and just past a 64-cell
chunk, patches with and without the logarithm table (above 2^19 cells), with and
without nested cells (levels 3: relativeToBottom 1, 2 and 4), behind and ahead
of a pulse.  The compensated sums agree with the ordered ones."""
import numpy as np
import pytest

import veritas_amd as va
from _amr_cases import two_slab_laser
from _oracle import OracleRun
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu

SHAPES = [(1, 8, 8), (1, 10, 62), (1, 34, 64), (1, 30, 66), (1, 12, 128), (1, 1026, 510), (1, 1026, 514),
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
