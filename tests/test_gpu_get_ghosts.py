"""Run.get and Run.patch with ghost layers: f slots with 0, 1 or 2, other planes also
with a part of the interior (negative); anything else is refused, also when only
the size is asked for."""
import numpy as np
import pytest

import veritas_amd as va

pytestmark = pytest.mark.gpu


def test_ghost_layers_of_every_kind_of_plane():
    p = va.two_stream(nx=24, np=40)
    r = va.Run(p, fused=False)
    r.advance(r.calc_dt(0.4), 2)
    for what in ("FxDS", "FpH3", "Cx"):
        full = r.get(what, 2)
        assert full.shape == (28, 44) and np.abs(full).max() > 0
        for g in (1, 0, -1, -5):
            want = full[2 - g:26 + g, 2 - g:42 + g]
            assert np.array_equal(r.get(what, g), want)
            assert np.array_equal(r.patch(0, 0, what, g), want)
    assert r.get("FxDS", -12).shape == (0, 16)
    size = va.host_lib().vxh_get
    for what, g in (("f1", 3), ("f1", -1), ("f0", -1), ("FxDS", 3), ("FxDS", -13)):
        for get in (lambda: r.get(what, g), lambda: r.patch(0, 0, what, g)):
            with pytest.raises(va.VeritasError, match="ghost"):
                get()
        assert size(r.h, what.encode(), g, None, 0) == -1
    r.close()
