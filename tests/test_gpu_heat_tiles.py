"""The heat field's loss and gradient at the edges of its tiles (32 x 32 results a wave, patches of 8 x 4
rows, runs of columns that span rows of voxels and segments of steps) against the 64-bit sums written
out here.

Tolerances, from the FP32 arithmetic: a rise is a sum of 26 products whose factors carry a few
roundings, so its error is at most 40 eps sum_q |A_q G_q| (eps = 2^-24), and likewise those of its
derivatives; an indicator's error is its slope, s (1 - s)/width, times that, plus 4 eps.  They are
propagated through the loss and the gradient term by term and summed without cancellation.
"""
import math

import numpy as np
import pytest

import amcafe_amd
from amcafe_amd.heat import HeatBatch, HeatField, track_desc

pytestmark = pytest.mark.gpu

TARGET = (220.0, 0.9, 0.4, 45e-6)
START = (200.0, 0.8, 0.35, 50e-6)
EPS = 2.0 ** -24
NONE = 1e-30  # terms that are skipped: below 2e-35 each


def _field(d, theta, nsteps):
    P, v, eta, sigma = theta
    xi, w = np.polynomial.legendre.leggauss(25)
    h = d.t_hist / 2
    tau, W = h * (1 - xi), h * w
    x, y, z = (((np.arange(n) + .5) * d.dX) for n in d.nX)
    t = (np.arange(nsteps) + 1) * d.dt
    C = eta * P / (math.pi * (d.k / d.alpha) * math.sqrt(4 * math.pi * d.alpha))
    A = 2 * d.alpha * tau + sigma ** 2
    D1 = 2 * A
    dy2 = np.tile((y - d.y_track) ** 2, len(z))[:, None]
    dz2 = np.repeat((z - d.z_track) ** 2, len(y))[:, None]
    a = W * C / (np.sqrt(tau) * A) * np.exp(-dy2 / D1 - dz2 / (4 * d.alpha * tau))
    tt = np.repeat(t, len(x))[:, None]
    dx = np.tile(x, len(t))[:, None] - d.x_start - v * (tt - tau)
    g = np.exp(-dx * dx / D1)
    gv = g * dx * (tt - tau) * 2 / D1
    rise, dv = a @ g.T, a @ gv.T
    ds = (a * (-2 * sigma / A + 4 * sigma / D1 ** 2 * dy2)) @ g.T + a @ (g * 4 * sigma / D1 ** 2 * dx * dx).T
    abs_v = a @ np.abs(gv).T
    abs_s = (a * (2 * sigma / A + 4 * sigma / D1 ** 2 * dy2)) @ g.T + a @ (g * 4 * sigma / D1 ** 2 * dx * dx).T
    return rise, dv, ds, abs_v, abs_s


def _expected(d, theta, target, nsteps):
    rise, dv, ds, abs_v, abs_s = _field(d, theta, nsteps)
    other = _field(d, target, nsteps)[0]
    ind = lambda r: 1 / (1 + np.exp(-np.clip((d.T0 - d.tL + r) / d.width, -700, 700)))
    a, b = ind(rise), ind(other)
    sa, sb = a * (1 - a), b * (1 - b)
    ea = sa / d.width * (40 * EPS * rise + 2 * EPS * d.tL) + 4 * EPS * a
    eb = sb / d.width * (40 * EPS * other + 2 * EPS * d.tL) + 4 * EPS * b
    lam, elam = 2 * (a - b) * sa / d.width, 2 / d.width * (sa * (ea + eb) + np.abs(a - b) * (ea + 4 * EPS * sa))
    grad, egrad = [], []
    for deriv, size in ((rise / theta[0], rise / theta[0]), (dv, abs_v), (rise / theta[2], rise / theta[2]), (ds, abs_s)):
        grad.append((lam * deriv).sum())
        egrad.append((elam * np.abs(deriv) + np.abs(lam) * 40 * EPS * size).sum())
    return ((a - b) ** 2).sum(), (2 * np.abs(a - b) * (ea + eb) + (ea + eb) ** 2).sum(), np.array(grad), np.array(egrad)


@pytest.mark.parametrize("nX,steps,checkpoint", [((1, 1, 1), 3, 100), ((1, 40, 30), 50, 16), ((2, 17, 9), 61, 100),
                                                 ((31, 15, 33), 33, 10), ((32, 32, 4), 64, 64), ((33, 31, 7), 40, 100),
                                                 ((65, 33, 9), 25, 7), ((100, 16, 8), 7, 3), ((48, 8, 16), 0, 5)])
def test_loss_and_gradient_at_the_tiles_edges(nX, steps, checkpoint):
    d = track_desc(nX, steps=max(steps, 1), checkpoint=checkpoint)
    l32, g32, _ = HeatField(d, TARGET).loss_grad_f32(START, 0, steps)
    only, _ = HeatField(d, TARGET).loss_f32(START, 0, steps)
    l64, _ = HeatField(d, TARGET).loss_f64(START, 0, steps)
    want, tol, grad, egrad = _expected(d, START, TARGET, steps)
    assert abs(l64 - want) <= 1e-9 * want + NONE, (l64, want)
    assert abs(l32 - want) <= tol + 4 * EPS * want + NONE, (l32, want, tol)
    assert only == l32
    for q in range(4):
        assert abs(g32[q] - grad[q]) <= egrad[q] + 4 * EPS * abs(grad[q]) + NONE, (q, g32[q], grad[q], egrad[q])
    # an instance of a batch has the bits of a call of its own
    loss, g, _ = HeatBatch(d, [TARGET, START, TARGET]).loss_grad_f32([START, TARGET, START], 0, steps)
    assert loss[0] == loss[2] == l32 and list(g[0]) == list(g[2]) == list(g32)


def test_parameters_that_are_not_finite_go_through():
    d = track_desc((33, 20, 9), steps=10)
    for q in range(4):
        theta = list(START)
        theta[q] = float("nan")
        loss, grad, _ = HeatField(d, TARGET).loss_grad_f32(theta, 0, 10)
        assert math.isnan(loss) and all(math.isnan(x) for x in grad), (q, loss, grad)
