"""States uploaded on their own (no other field) right before a step, with the liquid in planes that held none:
the marks of the planes that may hold liquid and the validity of the temperature field are reset with
them, in order with the step that follows.  Every field against the oracle, bit for bit."""
import numpy as np
import pytest

import amcafe_amd
from oracle_util import Oracle, tiny_deck

pytestmark = pytest.mark.gpu

NX, DX = (72, 64, 24), 2.5e-6
MELT = (1e-7, 1e-7, 1e-7, 1e-7)  # no voxel melts


def test_liquid_moves_between_steps():
    nxy, N = NX[0] * NX[1], NX[0] * NX[1] * NX[2]
    delt = 1e-9  # few captures
    o = Oracle(tiny_deck(NX, bmDelT=repr(delt), meltparam=MELT), crmath=True, bare=True)
    k = np.arange(N) // nxy
    f = dict(gID=(1 + np.arange(N) // 7 % 4).astype(np.int32), vState=np.full(N, 3, np.int32), extents=np.zeros(N),
             centroidOct=np.zeros(3 * N), BuildjID=np.zeros(N, np.int32))
    ct = np.array([0.3, 0.6, 0.0, 0.8] * 4)
    o.set_fields(TempCurr=np.full(N, 300.0), **f)
    o.set_grains(ct)
    o.L.orc_set_laser(o.h, 0, NX[2] - 1, 7)
    at = o.laser_inputs()
    dom = amcafe_amd.Domain(list(NX), DX, 1733.0, 1705.856, 300.0, list(MELT), 0.8, delt, 0.0, 2e-5, 3.0)
    dom.upload(**f)
    dom.set_grains(ct)
    rng = np.random.default_rng(5)
    for step, plane in enumerate((4, 17, 9, 21, 2, 13)):
        vs = np.full(N, 3, np.int32)
        vs[rng.choice(nxy, 40, replace=False) + plane * nxy] = 1
        dom.upload(vState=vs)
        o.set_fields(vState=vs)
        dom.temperature(*at)
        o.temperature()
        dom.update_voxels(7 + step, at[5])
        o.L.orc_set_laser(o.h, 0, NX[2] - 1, 7 + step)
        o.update_voxels()
        g, want = dom.download(), o.fields()
        assert (want["vState"] == 2).sum() > 100
        for key in ("gID", "vState", "extents", "centroidOct", "TempCurr", "BuildjID"):
            assert np.array_equal(g[key], want[key], equal_nan=want[key].dtype.kind == "f"), (step, key)
