"""The passes over the grid on rows of any length against the oracle: SetLiquid3, ConvertSolid1
(S/VoxelsCA.C:739-797) and the active set (S/VoxelsCA.C:262-303) of random states on domains whose
rows are shorter than, equal to and just beyond a thread's run of 16 voxels, so that runs span rows,
planes and the domain's end.  States, grains and counters are integers: the tolerance is zero.
"""
import numpy as np
import pytest

import amcafe_amd
from oracle_util import Oracle, tiny_deck

pytestmark = pytest.mark.gpu

DX, TL, TS = 2.5e-6, 1733.0, 1705.856
DELT = 0.05 * DX / 0.8


@pytest.mark.parametrize("nx", [(1, 1, 3), (1, 19, 5), (2, 7, 9), (3, 5, 4), (7, 3, 40), (15, 4, 5), (16, 3, 5), (17, 2, 6),
                                (16, 1, 7), (31, 9, 5), (33, 1, 8), (48, 24, 3), (50, 11, 6), (127, 10, 4)])
def test_grid_passes_on_rows_of_any_length(nx):
    N = nx[0] * nx[1] * nx[2]
    rng = np.random.default_rng(N)
    melt = (10e-6, 12e-6, 8e-6, 6e-6)
    for fill in (0.02, 0.4):  # few liquid voxels; many of every state
        vs = rng.choice([1, 2, 3], N, p=[fill, fill / 2, 1 - 1.5 * fill]).astype(np.int32)
        gid = np.where(vs >= 2, rng.integers(1, 4, N), 0).astype(np.int32)
        k, j, i = np.unravel_index(np.arange(N), (nx[2], nx[1], nx[0]))
        cen = ((np.stack([i, j, k], 1) + .5) * DX).reshape(-1)
        fields = dict(gID=gid, vState=vs, extents=np.where(vs >= 2, rng.uniform(0, 0.4, N) * DX, 0.0), centroidOct=cen,
                      BuildjID=np.zeros(N, np.int32))
        ct = np.array([0.0, 1.0, 0.0, 0.0, 0.3, 0.6, 0.0, 0.8, 0.7, 0.0, 0.6, 0.8])
        deck = tiny_deck(nx, bmDelT=repr(DELT), meltparam=melt)  # (a short step: few events)
        o = Oracle(deck, crmath=True, bare=True)
        o.set_fields(TempCurr=np.full(N, 300.0), **fields)
        o.set_grains(ct)
        o.L.orc_set_laser(o.h, 15 * nx[0], nx[2] - 1, 7)
        x, y, z, dirp, gth, il = o.laser_inputs()
        dom = amcafe_amd.Domain(list(nx), DX, TL, TS, 300.0, list(melt), 0.8, DELT, 0.0, 2e-5, 3.0)
        dom.upload(**fields)
        dom.set_grains(ct)
        for step in range(2):
            any_melt = dom.temperature(x, y, z, dirp, gth, il)
            o.temperature()
            st = dom.update_voxels(7, il)
            o.update_voxels()
            g, of, so = dom.download(), o.fields(), o.stats()
            assert any_melt == int(np.any(of["TempCurr"] >= TL))
            for key in ("TempCurr", "vState", "gID", "BuildjID", "extents", "centroidOct"):
                assert np.array_equal(g[key], of[key], equal_nan=of[key].dtype.kind == "f"), (fill, step, key)
            for key in ("n_active", "n_events"):
                assert st[key] == so[key], (fill, step, key)
