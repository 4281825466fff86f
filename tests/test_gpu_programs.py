"""The task programs of a hierarchy with few patches (the workgroups read their
LDS copy of the patch table) and with more (the table itself), bit for bit
against the oracle."""
import pytest

import veritas_amd as va
from _amr_cases import two_slab_laser
from _oracle import OracleRun
from test_gpu_amr import compare_fields, compare_mesh

pytestmark = pytest.mark.gpu


def few():
    return va.laser(nx=384, np=64, levels=3, wavelengths=24.0, ramp=6.0, fwhm_cycles=3.0)


@pytest.mark.parametrize("make,most", [(few, True), (two_slab_laser, False)], ids=["few", "many"])
def test_hierarchy_matches_the_oracle(make, most):
    p = make()
    g, o = va.Run(p), OracleRun(p)
    n = len(g.layout())
    print(f"case: {n} patches", flush=True)
    assert (2 <= n <= 12) if most else n > 12
    dt = o.calc_dt(0.4)
    g.advance(dt, 2)
    o.advance(dt, 2)
    compare_mesh(g, o, "two steps")
    compare_fields(g, o, "two steps")
    g.close()
    o.close()
