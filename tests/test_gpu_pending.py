"""A batch in which one deck's nucleation pool runs out in the very step in which another deck's growing
list outgrows the capture tier: the larger tier relaunches the loop for all of them before the pool is
refilled, and the suspended nucleation has to wait for its own orientation (S/VoxelsCA.C:483-505)."""
import re

import numpy as np
import pytest

import amcafe_amd
from oracle_util import read

pytestmark = pytest.mark.gpu

TIERS = (1024, 2048, 4096, 8192)
DECKS = [("t_odd.in", "3e-3"), ("c2_batched/inst_44.in", "1e-3"), ("c2_batched/inst_24.in", "1e-3")]
STEPS = 90


def test_a_pending_nucleation_waits_for_its_pool(monkeypatch):
    decks = [re.sub(r"(?m)^r .*$", f"r {r}", read(name)) for name, r in DECKS]
    monkeypatch.setenv("AMCAFE_POOL_CHUNK", "1")
    batch = amcafe_amd.Sim(decks)
    cap, last, both = TIERS[1], [0] * len(decks), 0
    for _ in range(STEPS):
        batch.step()
        st = [batch.stats(i) for i in range(len(decks))]
        grown = any(s["n_growing"] > cap for s in st)
        empty = any(s["n_nucleations"] > 1 + 2 * n for s, n in zip(st, last) if s["n_growing"] <= cap)
        both += grown and empty
        last = [s["n_nucleations"] for s in st]
        most = max(s["n_growing"] for s in st)
        cap = next(t for t in TIERS if t >= most + most // 32)
    assert both > 0
    monkeypatch.delenv("AMCAFE_POOL_CHUNK")
    for i, deck in enumerate(decks):
        one = amcafe_amd.Sim(deck)
        one.run(STEPS)
        assert one.info(0)["tInd"] == batch.info(i)["tInd"]
        f, g = batch.fields(i), one.fields(0)
        for k in f:
            assert np.array_equal(f[k], g[k], equal_nan=f[k].dtype.kind == "f"), (DECKS[i], k)
        assert np.array_equal(batch.grains(i), one.grains(0)), DECKS[i]
