"""The base plate's and the first powder layer's Voronoi grains (S/BasePlate.C:74-117,
S/VoxelsCA.C:125-161, 920-981) on domains that are no multiple of the kernel's 8x8x4 bricks and with
site counts around its groups of 256, against the oracle's search over all sites.  Grain ids and states are
integers and the centroids voxel centres: the tolerance is zero."""
import numpy as np
import pytest

import amcafe_amd
from oracle_util import Oracle, tiny_deck

pytestmark = pytest.mark.gpu

DX = 2.5e-6


@pytest.mark.parametrize("nx,plate,layer,grains", [((3, 2, 9), 4, 2, 3), ((8, 8, 8), 4, 2, 40), ((9, 17, 11), 5, 3, 250),
                                                   ((33, 7, 14), 9, 2, 300), ((65, 24, 8), 3, 4, 700),
                                                   ((16, 40, 21), 13, 5, 520)])
def test_initial_grains(nx, plate, layer, grains):
    mu = grains / (nx[0] * nx[1] * plate * 2.5 ** 3)
    deck = tiny_deck(nx, mu=repr(mu), lrate=repr(mu), bpH=repr(plate * DX), lT=repr(layer * DX))
    sim, o = amcafe_amd.Sim(deck), Oracle(deck, crmath=True)
    f, of = sim.fields(0), o.fields()
    for key in ("gID", "vState", "centroidOct", "extents"):
        assert np.array_equal(f[key], of[key], equal_nan=of[key].dtype.kind == "f"), key
    assert np.array_equal(sim.grains(0), o.grains())
