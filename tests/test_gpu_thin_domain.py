"""The base plate's grains (S/BasePlate.C:74-117) of a domain one voxel wide and 67.2 million high: as many
bricks of the search as a quarter of its voxels, more than one launch can give a workgroup each (256
threads a brick: past 2^32).  Against the nearest of all sites, first of equals, with the reference's
squared distance."""
import numpy as np
import pytest

import amcafe_amd
from oracle_util import initial_sites, tiny_deck

pytestmark = pytest.mark.gpu

NZ, DX = 67_200_000, 2.5e-6


def test_plate_of_a_column():
    plate = NZ - 4
    deck = tiny_deck((1, 1, NZ), mu=repr(40 / (2.5 ** 3 * NZ)), lrate="0.1", bpH=repr(plate * DX), lT=repr(2 * DX))
    xp, _, _, _, nzh, iz1, _ = initial_sites(deck)
    assert 4 < len(xp) < 200 and nzh > 2 ** 26
    sim = amcafe_amd.Sim(deck)
    gid = sim.fields(0, which=("gID",))["gID"]
    sim.close()
    top = min(nzh, iz1)
    for k0 in range(0, top, 1 << 23):
        z = (np.arange(k0, min(top, k0 + (1 << 23))) + .5) * DX
        best, bd = np.zeros(z.size, np.int32), np.full(z.size, np.inf)
        for q, (sx, sy, sz) in enumerate(xp):
            ax, ay, az = .5 * DX - sx, .5 * DX - sy, z - sz
            d = ax * ax + ay * ay + az * az
            lt = d < bd
            best[lt], bd[lt] = q + 1, d[lt]
        assert np.array_equal(gid[k0:k0 + z.size], best), k0
