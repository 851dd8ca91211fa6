"""amcafe_heat_last_evaluations after each kind of call: the FP64 loss evaluates every voxel at every
step; the FP32 calls at most that, and all of it where the whole domain is near the track."""
import pytest

import amcafe_amd
from amcafe_amd.heat import HeatField, track_desc

pytestmark = pytest.mark.gpu

TARGET = (220.0, 0.9, 0.4, 45e-6)
START = (200.0, 0.8, 0.35, 50e-6)


@pytest.mark.parametrize("nX,steps,checkpoint", [((33, 31, 7), 41, 10), ((1, 1, 1), 3, 100), ((48, 8, 16), 0, 5)])
def test_evaluations_are_counted(nX, steps, checkpoint):
    f = HeatField(track_desc(nX, steps=max(steps, 1), checkpoint=checkpoint), TARGET)
    evals = amcafe_amd.lib().amcafe_heat_last_evaluations
    total = steps * nX[0] * nX[1] * nX[2]
    f.loss_f64(START, 0, steps)
    assert evals() == total
    f.loss_f32(START, 0, steps)
    some = evals()
    assert 0 <= some <= total
    f.loss_grad_f32(START, 0, steps)
    assert evals() == some
    f.loss_f64(START, 0, steps)
    assert evals() == total
