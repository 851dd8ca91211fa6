"""A flat front of more than a thousand growing cells whose first captures tie in time exactly (unrotated
grains, dx a power of two), above a front of its own further on whose cells do not: the windows fall back to one
event each for hundreds of events and go on with wide ones afterwards.  Every field and counter against
the oracle, bit for bit."""
import functools

import numpy as np
import pytest

import amcafe_amd
from oracle_util import Oracle, tiny_deck
from test_gpu_capture_windows import AVEL, DX, MELT, NVEL, TL, TS, VHAT

pytestmark = pytest.mark.gpu

NX = (37, 31, 7)


@functools.lru_cache(maxsize=None)
def _expected():
    nxy, N = NX[0] * NX[1], NX[0] * NX[1] * NX[2]
    k = np.arange(N) // nxy
    vs = np.where((k == 0) | (k == 6), 2, 1).astype(np.int32)  # two flat fronts
    ext = np.where(k == 0, 0.5 * DX, 0.0)                      # the lower one's captures tie
    ext[k == 6] = (np.arange(nxy) * 7919 % 1009) / 1009 * 0.3 * DX
    j, i = np.arange(N) % nxy // NX[0], np.arange(N) % NX[0]
    f = dict(gID=np.where(k == 0, 1, np.where(k == 6, 2 + np.arange(N) % 2, 0)).astype(np.int32), vState=vs, extents=ext,
             centroidOct=((np.stack([i, j, k], 1) + .5) * DX).reshape(-1), BuildjID=np.zeros(N, np.int32))
    ct = np.array([0.0, 1.0, 0.0, 0.0, 0.3, 0.6, 0.0, 0.8, 0.7, 0.0, 0.6, 0.8])
    delt = 0.75 * DX / VHAT
    o = Oracle(tiny_deck(NX, dx=repr(DX), r="0", bmDelT=repr(delt), meltparam=MELT), crmath=True, bare=True)
    o.set_fields(TempCurr=np.full(N, 300.0), **f)
    o.set_grains(ct)
    o.L.orc_set_laser(o.h, 0, NX[2] - 1, 7)
    at = o.laser_inputs()
    o.temperature()
    o.update_voxels()
    return f, ct, at, delt, o.fields(), o.stats(), o.events()[2]


@pytest.mark.parametrize("tier", [0, 1, 2, 3, 4, 5])
def test_ties_then_ordinary_growth(monkeypatch, tier):
    monkeypatch.setenv("AMCAFE_CAPTURE_TIER_MIN", str(tier))
    fields, ct, at, delt, of, so, dt = _expected()
    assert (dt[1:] == 0).sum() > 1000 and (dt > 0).sum() > 200  # both kinds
    dom = amcafe_amd.Domain(list(NX), DX, TL, TS, 300.0, list(MELT), 0.8, delt, 0.0, AVEL, NVEL)
    dom.upload(**fields)
    dom.set_grains(ct)
    dom.temperature(*at)
    st = dom.update_voxels(7, at[5])
    g = dom.download()
    for key in ("n_active", "n_events", "n_captures"):
        assert st[key] == so[key], f"{key} {st[key]} vs {so[key]}"
    for key in ("gID", "vState", "TempCurr", "extents", "centroidOct"):
        assert np.array_equal(g[key], of[key], equal_nan=key in ("extents", "centroidOct")), key
