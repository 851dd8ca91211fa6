"""The capture loop's work counters on a step of one event: a flat front of 1,147 cells ties for it, so a scan
has to look at every one of them (slot_visits), at one capture time of each at least (cand_evals), and
no scan looks at a cell twice."""
import numpy as np
import pytest

import amcafe_amd
from test_gpu_capture_windows import AVEL, DX, MELT, NVEL, TL, TS, VHAT

pytestmark = pytest.mark.gpu

NX = (37, 31, 5)


@pytest.mark.parametrize("tier", [0, 1, 2, 3, 4, 5])
def test_scans_count_cells_and_times(monkeypatch, tier):
    monkeypatch.setenv("AMCAFE_CAPTURE_TIER_MIN", str(tier))
    nxy, N = NX[0] * NX[1], NX[0] * NX[1] * NX[2]
    k, j, i = np.unravel_index(np.arange(N), (NX[2], NX[1], NX[0]))
    dom = amcafe_amd.Domain(list(NX), DX, TL, TS, 300.0, list(MELT), 0.8, 0.1 * DX / VHAT, 0.0, AVEL, NVEL)
    dom.upload(gID=(k == 0).astype(np.int32), vState=np.where(k == 0, 2, 1).astype(np.int32), extents=(k == 0) * 0.5 * DX,
               centroidOct=((np.stack([i, j, k], 1) + .5) * DX).reshape(-1), BuildjID=np.zeros(N, np.int32))
    dom.set_grains(np.array([0.0, 1.0, 0.0, 0.0]))
    dom.temperature(0.0, 0.0, (NX[2] - 1) * DX, 1.0, 0.0, NX[2] - 1)
    st = dom.update_voxels(7, NX[2] - 1)
    assert st["n_events"] == 1 and st["n_active"] == N
    # (four ways of filling a window, and a last window that finds the step's time used up)
    assert nxy <= st["slot_visits"] <= 8 * st["n_growing"], st
    assert st["slot_visits"] + 1 <= st["cand_evals"] <= 27 * st["slot_visits"] + 128, st
