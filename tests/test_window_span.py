"""The clock span of the capture loop's windows, as the kernel adapts it (the same function on the host):
however long the windows hold ties or a few cells only, it stays within a range from which the next
windows recover.  Unbounded, it went to zero after 799 tied windows of a 1e-6 s step, to infinity (in
single precision) after 216 with a few heads, and stayed there."""
import ctypes

import pytest

import amcafe_amd


def _span():
    f = amcafe_amd.lib().amcd_window_span
    f.restype, f.argtypes = ctypes.c_double, [ctypes.c_double, ctypes.c_int, ctypes.c_int, ctypes.c_double, ctypes.c_int]
    return f


@pytest.mark.parametrize("DelT", [1e-9, 3.125e-6, 1.0])
@pytest.mark.parametrize("cells", [0, 1, 300, 15000, 10 ** 7])
@pytest.mark.parametrize("bins,mode", [(0, 0), (0, 1), (0, 2), (0, 3), (32, 0), (32, 1)])
def test_span_stays_in_range_and_recovers(DelT, cells, bins, mode):
    f = _span()
    first = span = f(-1.0, 0, 0, DelT, cells)
    assert 0 < first <= DelT
    for _ in range(5000):
        span = f(span, bins, mode, DelT, cells)
        assert first / 1024 <= span <= 64 * DelT
    if mode >= 2:
        assert span == first
    n = 0  # windows until it is back where it began, with as few or as many heads as that takes
    while not 0.3 * first <= span <= 3 * first:
        span = f(span, 32 if span < first else 0, 0, DelT, cells)
        n += 1
    assert n <= 20


def test_ordinary_windows_adapt_as_before():
    f = _span()
    for bins, want in [(0, 0.4), (2, 0.4), (5, 0.5), (18, 1.0), (31, 1.5), (32, 1.6)]:
        assert abs(f(1e-7, bins, 0, 1e-6, 300) / 1e-7 - want) < 1e-12
