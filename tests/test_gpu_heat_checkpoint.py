"""The heat field with segments longer than the call, short last segments and one-step segments, against the
64-bit sums and tolerances of test_gpu_heat_tiles.  A checkpoint beyond the call's length is the call's
length: the same bits."""
import ctypes

import pytest

import amcafe_amd
from amcafe_amd.heat import HeatField, track_desc
from test_gpu_heat_tiles import EPS, NONE, START, TARGET, _expected

pytestmark = pytest.mark.gpu


def _noalloc(d, steps):
    th, tg = (ctypes.c_double * 4)(*START), (ctypes.c_double * 4)(*TARGET)
    loss, grad = (ctypes.c_double * 1)(), (ctypes.c_double * 4)()
    rc = amcafe_amd.lib().amcafe_heat_loss_grad_batch_f32_noalloc(ctypes.byref(d), 1, th, tg, 0, steps, loss, grad)
    assert rc == 0
    return loss[0], list(grad)


@pytest.mark.parametrize("nX,steps,checkpoint", [((64, 1, 4), 30, 2 ** 31 - 1), ((128, 1, 1), 20, 2 ** 30),
                                                 ((64, 32, 16), 20, 2 ** 31 - 1), ((33, 31, 7), 40, 1000),
                                                 ((65, 33, 9), 25, 24), ((32, 17, 9), 5, 1)])
def test_any_checkpoint(nX, steps, checkpoint):
    d = track_desc(nX, steps=steps, checkpoint=checkpoint)
    f = HeatField(d, TARGET)
    l32, g32, _ = f.loss_grad_f32(START, 0, steps)
    l64, _ = f.loss_f64(START, 0, steps)
    want, tol, grad, egrad = _expected(d, START, TARGET, steps)
    assert abs(l64 - want) <= 1e-9 * want + NONE, (l64, want)
    assert abs(l32 - want) <= tol + 4 * EPS * want + NONE, (l32, want, tol)
    for q in range(4):
        assert abs(g32[q] - grad[q]) <= egrad[q] + 4 * EPS * abs(grad[q]) + NONE, (q, g32[q], grad[q], egrad[q])
    assert f.loss_f32(START, 0, steps)[0] == l32
    assert _noalloc(d, steps) == (l32, list(g32))
    if checkpoint > steps:
        e = HeatField(track_desc(nX, steps=steps, checkpoint=steps), TARGET)
        assert e.loss_grad_f32(START, 0, steps)[:2] == (l32, g32)
        assert e.loss_f64(START, 0, steps)[0] == l64
