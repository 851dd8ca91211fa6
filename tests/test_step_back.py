"""How far the capture loop's clock may step back before a cell's half-diagonal is zero (the kernel's function
on the host): a number for every cell, never more than e/v by the part in 2^16 that the loop takes off
it, and no limit only for cells that do not grow."""
import ctypes
import math

import pytest

import amcafe_amd


@pytest.mark.parametrize("v", [0.0, 5e-324, 1e-300, 1e-46, 1e-45, 1e-40, 1e-38, 1e-31, 1.1e-30, 1e-12, 0.5, 3e38])
@pytest.mark.parametrize("e", [0.0, 5e-324, 1e-60, 1e-46, 1e-44, 1e-38, 1e-12, 1e-6, 1.0])
def test_a_bound_for_every_cell(e, v):
    f = amcafe_amd.lib().amcd_step_back
    f.restype, f.argtypes = ctypes.c_float, [ctypes.c_double, ctypes.c_double]
    x = f(e, v)
    if v == 0.0:
        assert x == math.inf
        return
    assert x == x and x >= 0.0
    # (below single precision's normal range a product may round up: by less than 2^-149)
    assert x * (1 - 2.0 ** -16) <= e / v + 2.0 ** -149, (e, v, x)
    if e / v < 1e37 and v > 1e-30 and e > 1e-37:
        assert x >= e / v * (1 - 2.0 ** -20) or e / v < 1e-37
