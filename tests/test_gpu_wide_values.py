"""Values of f beyond the range of the short division sequences (WENO_MAX =
2^190 in vx_dev.h): wavefronts that meet one take the full-range form, the
others the short one.  A reference density that puts the bulk of f above the
limit and its tails below it drives both, and the result is the oracle's bit
for bit (the operations are IEEE divisions either way)."""
import numpy as np
import pytest

import veritas_amd as va
from _amr_cases import two_slab_laser
from _oracle import OracleRun
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu

LIMIT = 2.0 ** 190

CASES = [
    ("landau fused 64x256", va.landau(n_ref=1e38), True),
    ("landau sub-steps 64x256", va.landau(n_ref=1e38), False),
    ("landau fused 150x131, many strips", va.landau(nx=150, np=132, n_ref=1e38), True),
    ("laser single level, pulse", two_slab_laser(levels=1, lambda0=1e-13), True),
    ("laser two levels", two_slab_laser(levels=2, lambda0=1e-13), True),
]


@pytest.mark.parametrize("name,p,fused", CASES, ids=[c[0] for c in CASES])
def test_values_beyond_the_short_divisions(name, p, fused):
    print(f"case: {name}", flush=True)
    g, o = va.Run(p, fused=fused), OracleRun(p)
    f = o.get("f1")
    assert f.max() > LIMIT and f[f > 0].min() < LIMIT
    dt = o.calc_dt(0.4)
    assert g.calc_dt(0.4) == dt
    g.advance(dt, 2)
    o.advance(dt, 2)
    lay = o.layout()
    assert np.array_equal(g.layout(), lay)
    for lvl in sorted(set(lay[:, 0])):
        for k in range(int((lay[:, 0] == lvl).sum())):
            a, b = g.patch(lvl, k, "f1"), o.patch(lvl, k, "f1")
            assert np.isfinite(b).all()
            assert_same(f"{name} level {lvl} patch {k}", a, b)
    g.close()
    o.close()
