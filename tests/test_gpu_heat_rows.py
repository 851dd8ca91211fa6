"""The heat field on the longest row of voxels that its arguments allow (2^31 - 1): 2^24 groups of rows, whose
threads a launch must not count past 2^32.  Only a band around the track is warm, so the sums are those of
that band alone (64-bit, written out in test_gpu_heat_tiles).  At 2.7 km from the origin a position is good to
6e-13 m, which moves an exponent by at most 2 dy 6e-13/D1 = 1e-7 and the indicators by 1e-5 of themselves:
tolerance 1e-4 (1e-3 for the gradient's sums, whose terms cancel in part), besides FP32's own."""
import pytest

from amcafe_amd.heat import HeatField, track_desc
from test_gpu_heat_tiles import START, TARGET, _expected

pytestmark = pytest.mark.gpu


def test_the_longest_row():
    N, band = 2 ** 31 - 1, 1601  # (the same voxel in the middle of both)
    f = HeatField(track_desc((1, N, 1), steps=1), TARGET)
    want, tol, grad, egrad = _expected(track_desc((1, band, 1), steps=1), START, TARGET, 1)
    assert want > 0.1
    l32, g32, _ = f.loss_grad_f32(START, 0, 1)
    assert abs(l32 - want) <= tol + 1e-4 * want, (l32, want)
    for q in range(4):
        assert abs(g32[q] - grad[q]) <= egrad[q] + 1e-3 * abs(grad[q]), (q, g32[q], grad[q], egrad[q])
    l64, _ = f.loss_f64(START, 0, 1)
    assert abs(l64 - want) <= 1e-4 * want, (l64, want)
