"""The capture loop's windows (S/VoxelsCA.C:381-610) at their edges, against the oracle: states in
which many candidates tie exactly in time (unrotated grains and dx a power of two, so that a window
holds one event's worth of clock and is overfull), captures that follow each other within one clock
value, half-diagonals beyond the capture distance (negative times: the clock steps back and
half-diagonals clamp at zero), and nucleation.  Every field and counter of a step: a difference of one
bit would mean another event order, so the tolerance is zero.
"""
import functools

import numpy as np
import pytest

import amcafe_amd
from oracle_util import Oracle, tiny_deck

pytestmark = pytest.mark.gpu

DX = 2.0 ** -18
TL, TS, AVEL, NVEL = 1733.0, 1705.856, 2e-5, 3.0
VHAT = AVEL * (TL - TS) ** NVEL
MELT = (1e-7, 1e-7, 1e-7, 1e-7)  # no voxel melts
NX = (13, 11, 8)


def _state(extent, every, rotated):
    nx, ny, nz = NX
    N = nx * ny * nz
    k, j, i = np.unravel_index(np.arange(N), (nz, ny, nx))
    seed = (i % every == 1) & (j % every == 1) & (k % every == 1)
    ids = np.flatnonzero(seed)
    vs = np.where(seed, 2, 1).astype(np.int32)
    vs[(i == nx - 1) & (j % 2 == 0)] = 3  # some solid, which turns mushy
    gid = np.where(vs >= 2, 1 + np.arange(N) % 3, 0).astype(np.int32)
    e = {"equal": 0.875, "mixed": None, "beyond": None}[extent]
    ext = np.zeros(N)
    lo, hi = (0.0, 1.0) if extent == "mixed" else (0.0, 1.5)
    ext[ids] = (e if e is not None else np.linspace(lo, hi, ids.size)[::-1]) * np.ones(ids.size) * DX
    cen = (np.stack([i, j, k], 1) + .5) * DX
    ct = np.array([0.0, 1.0, 0.0, 0.0] * 3) if not rotated else np.array(
        [0.0, 1.0, 0.0, 0.0, 0.3, 0.6, 0.0, 0.8, 0.7, 0.0, 0.6, 0.8])
    return dict(gID=gid, vState=vs, extents=ext, centroidOct=cen.reshape(-1), BuildjID=np.zeros(N, np.int32)), ct


CASES = [("equal", 3, False, 0.0, 0), ("equal", 3, True, 0.0, 2), ("mixed", 3, True, 2e-4, 0), ("beyond", 3, False, 1e-4, 2),
         ("beyond", 2, True, 0.0, 0), ("equal", 16, False, 0.0, 2),
         ("mixed", 3, True, 2e-2, 0)]  # every event nucleates: the pool of orientations is refilled over and over


@functools.lru_cache(maxsize=None)
def _expected(extent, every, rotated, r, above):
    """The oracle's step; `above`: planes over the laser's, at T0 (growth velocities far larger)."""
    delt = 1.2 * DX / VHAT
    o = Oracle(tiny_deck(NX, dx=repr(DX), r=repr(r), bmDelT=repr(delt), meltparam=MELT), crmath=True, bare=True)
    fields, ct = _state(extent, every, rotated)
    o.set_fields(TempCurr=np.full(o.N, 300.0), **fields)
    o.set_grains(ct)
    o.L.orc_set_laser(o.h, 0, NX[2] - 1 - above, 7)
    at = o.laser_inputs()
    o.temperature()
    o.update_voxels()
    return fields, ct, at, delt, o.fields(), o.stats(), o.grains()


@pytest.mark.parametrize("tier", [0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("case", CASES)
def test_windows_at_their_edges(monkeypatch, tier, case):
    monkeypatch.setenv("AMCAFE_CAPTURE_TIER_MIN", str(tier))
    fields, ct, at, delt, of, so, og = _expected(*case)
    dom = amcafe_amd.Domain(list(NX), DX, TL, TS, 300.0, list(MELT), 0.8, delt, case[3], AVEL, NVEL)
    dom.upload(**fields)
    dom.set_grains(ct)
    dom.temperature(*at)
    st = dom.update_voxels(7, at[5])
    g = dom.download()
    for key in ("n_active", "n_events", "n_captures", "n_nucleations"):
        assert st[key] == so[key], f"{key} {st[key]} vs {so[key]}"
    for key in ("gID", "vState", "TempCurr", "extents", "centroidOct"):
        assert np.array_equal(g[key], of[key], equal_nan=key in ("extents", "centroidOct")), key
    assert np.array_equal(dom.grains(), og), "grain table"
    assert st["n_events"] > 20
