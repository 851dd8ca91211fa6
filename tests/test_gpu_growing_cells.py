"""Steps in which far more of the active cells grow than the capture loop keeps records for (half of them;
records are sized for a quarter): the captures of the others are re-centred when they happen.  Every
field and counter against the oracle, bit for bit, in every capture tier."""
import functools

import numpy as np
import pytest

import amcafe_amd
from oracle_util import Oracle, tiny_deck
from test_gpu_capture_windows import AVEL, DX, MELT, NVEL, TL, TS, VHAT

pytestmark = pytest.mark.gpu

NX = (13, 11, 8)


@functools.lru_cache(maxsize=None)
def _expected(r, reach):
    """Every other plane of voxels mushy, with half-diagonals spread over [0, reach] and three rotations."""
    N = NX[0] * NX[1] * NX[2]
    k, j, i = np.unravel_index(np.arange(N), (NX[2], NX[1], NX[0]))
    mushy = k % 2 == 1
    f = dict(gID=np.where(mushy, 1 + np.arange(N) % 3, 0).astype(np.int32), vState=np.where(mushy, 2, 1).astype(np.int32),
             extents=np.where(mushy, (np.arange(N) * 7919 % 1000) / 1000 * reach * DX, 0.0),
             centroidOct=((np.stack([i, j, k], 1) + .5) * DX).reshape(-1), BuildjID=np.zeros(N, np.int32))
    ct = np.array([0.0, 1.0, 0.0, 0.0, 0.3, 0.6, 0.0, 0.8, 0.7, 0.0, 0.6, 0.8])
    delt = 0.9 * DX / VHAT
    o = Oracle(tiny_deck(NX, dx=repr(DX), r=repr(r), bmDelT=repr(delt), meltparam=MELT), crmath=True, bare=True)
    o.set_fields(TempCurr=np.full(N, 300.0), **f)
    o.set_grains(ct)
    o.L.orc_set_laser(o.h, 0, NX[2] - 1, 7)
    at = o.laser_inputs()
    o.temperature()
    o.update_voxels()
    return f, ct, at, delt, o.fields(), o.stats(), o.grains()


@pytest.mark.parametrize("tier", [0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("case", [(0.0, 0.9), (2e-4, 0.9), (2e-4, 1.3)])
def test_half_of_the_active_cells_grow(monkeypatch, tier, case):
    monkeypatch.setenv("AMCAFE_CAPTURE_TIER_MIN", str(tier))
    fields, ct, at, delt, of, so, og = _expected(*case)
    dom = amcafe_amd.Domain(list(NX), DX, TL, TS, 300.0, list(MELT), 0.8, delt, case[0], AVEL, NVEL)
    dom.upload(**fields)
    dom.set_grains(ct)
    dom.temperature(*at)
    st = dom.update_voxels(7, at[5])
    g = dom.download()
    assert st["n_growing"] > st["n_active"] // 4 + 100
    for key in ("n_active", "n_events", "n_captures", "n_nucleations"):
        assert st[key] == so[key], f"{key} {st[key]} vs {so[key]}"
    for key in ("gID", "vState", "TempCurr", "extents", "centroidOct"):
        assert np.array_equal(g[key], of[key], equal_nan=key in ("extents", "centroidOct")), key
    assert np.array_equal(dom.grains(), og), "grain table"
    assert st["n_events"] > 20
