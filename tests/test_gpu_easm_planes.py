"""EASM temperatures (S/TempField.C:79-137) that melt planes which held no liquid before, with no upload in
between: the laser goes up ten planes, so that ConvertSolid1 (S/VoxelsCA.C:780-797) has to find the liquid
where neither the last step nor an analytic evaluation had any.  A plane holds more voxels than a block
of the pass.  The device's temperatures are handed to the oracle; every field bit for bit."""
import numpy as np
import pytest

import amcafe_amd
from oracle_util import Oracle, tiny_deck

pytestmark = pytest.mark.gpu

NX, DX = (80, 56, 20), 2.5e-6
KEYS = ("gID", "vState", "extents", "centroidOct", "BuildjID")


def test_the_laser_goes_up_between_easm_steps():
    o = Oracle(tiny_deck(NX, r="1e-3", lT="10e-6"), crmath=True, bare=True)
    N = o.N
    k, j, i = np.unravel_index(np.arange(N), (NX[2], NX[1], NX[0]))
    f = dict(gID=(1 + (i // 9 + j // 7 * 3 + k // 5 * 5) % 5).astype(np.int32), vState=np.full(N, 3, np.int32),
             extents=np.zeros(N), centroidOct=((np.stack([i, j, k], 1) + .5) * DX).reshape(-1),
             BuildjID=np.zeros(N, np.int32))
    ct = np.array([0.3, 0.6, 0.0, 0.8] * 5)
    o.set_fields(TempCurr=np.full(N, 300.0), **f)
    o.set_grains(ct)
    dom = amcafe_amd.Domain(list(NX), DX, 1733.0, 1705.856, 300.0, [20e-6, 60e-6, 15e-6, 12e-6], 0.8, 3.125e-6, 1e-3,
                            2e-5, 3.0)
    dom.upload(**f)
    dom.set_grains(ct)
    events = 0
    for tind, (plane, x) in enumerate([(7, 60e-6), (7, 62e-6), (17, 64e-6), (17, 66e-6), (12, 90e-6), (12, 92e-6)], 7):
        dom.easm_temperature(x, -85e-6, plane * DX, 1.0, 0.0, plane, 200.0, 10e-6)
        g = dom.download()
        o.set_fields(TempCurr=g["TempCurr"], BuildjID=g["BuildjID"])
        o.L.orc_set_laser(o.h, 0, plane, tind)
        assert (g["TempCurr"] >= 1733.0).sum() > 100
        st = dom.update_voxels(tind, plane)
        o.update_voxels()
        g, want = dom.download(), o.fields()
        for key in KEYS:
            assert np.array_equal(g[key], want[key], equal_nan=g[key].dtype.kind == "f"), (tind, key)
        assert st["n_active"] == o.stats()["n_active"]
        events += st["n_events"]
    assert np.array_equal(dom.grains(), o.grains())
    assert events > 100
