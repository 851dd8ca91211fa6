"""EASM temperatures where the kernel hands voxels from threads to groups of 16 lanes: domains that are
no multiple of a workgroup, powers from one that leaves no voxel iterating (all done by the threads) to
ones that keep a shell of voxels going round the properties' jump at 1660 K for all 100 steps.
Against the oracle's restatement of TempField::EASM (S/TempField.C:79-137, S/Utilities.C:60-140):
temperatures within 1e-9 relative (FP64 throughout, another order of sums), flags and the number of source integrals equal -- the latter also
holds the count of the steps that a repeating iteration does not evaluate."""
import numpy as np
import pytest

import amcafe_amd
from oracle_util import Oracle, tiny_deck

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [(1, 1, 5), (37, 29, 11), (67, 5, 9), (128, 24, 4)])
@pytest.mark.parametrize("power", [20.0, 120.0, 200.0, 400.0])
def test_easm_threads_and_groups(nx, power):
    dx, lT = 2.5e-6, 5e-6
    deck = tiny_deck(nx, bmP=repr(power))
    o = Oracle(deck, crmath=False, bare=True)
    N = nx[0] * nx[1] * nx[2]
    o.set_fields(gID=np.zeros(N, np.int32), vState=np.full(N, 3, np.int32), TempCurr=np.full(N, 300.0),
                 extents=np.zeros(N), centroidOct=np.zeros(3 * N), BuildjID=np.zeros(N, np.int32))
    dom = amcafe_amd.Domain(list(nx), dx, 1733.0, 1705.856, 300.0, [20e-6, 60e-6, 15e-6, 12e-6], 0.8, 3.125e-6, 0.0,
                            2e-5, 3.0)
    il = nx[2] - 1
    for x, gth in ((0.6 * nx[0] * dx, 0.0), (0.9 * nx[0] * dx, 1.1693705988362009)):
        y, z = 0.5 * nx[1] * dx, il * dx
        alld, nd = dom.easm_temperature(x, y, z, 1.0, gth, il, power, lT)
        allo, no = o.easm(x, y, z, gth)
        g, f = dom.download(), o.fields()
        assert (alld, nd) == (allo, no)
        assert np.array_equal(g["BuildjID"], f["BuildjID"])
        np.testing.assert_allclose(g["TempCurr"], f["TempCurr"], rtol=1e-9, atol=0)
