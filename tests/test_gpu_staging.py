"""Temperatures asked for in a row without their end-of-scan flag (amcafe_analytic_temp_curr with a null
any_melt returns before the device has run): every one takes its own laser.  BuildjID keeps the union
of the melt pools (S/TempField.C:139-217), so a lost position shows; the same calls with the flag read back
are the expectation, and an EASM evaluation may follow as well."""
import ctypes

import numpy as np
import pytest

import amcafe_amd
from amcafe_amd._lib import Laser, check, lib

pytestmark = pytest.mark.gpu

NX, DX = (256, 192, 48), 2.5e-6


def _domain():
    N = NX[0] * NX[1] * NX[2]
    dom = amcafe_amd.Domain(list(NX), DX, 1733.0, 1705.856, 300.0, [10e-6, 20e-6, 15e-6, 12e-6], 0.8, 3.125e-6, 0.0, 2e-5,
                            3.0)
    dom.upload(gID=np.ones(N, np.int32), vState=np.full(N, 3, np.int32), extents=np.zeros(N), centroidOct=np.zeros(3 * N),
               BuildjID=np.zeros(N, np.int32))
    return dom


@pytest.mark.parametrize("easm", [False, True])
def test_temperatures_in_a_row(easm):
    a, b = _domain(), _domain()
    melted = 0
    for q in range(24):
        at = ((20 + 9 * q) * DX, (30 + 5 * q) * DX, (40 - q % 3) * DX, 1.0, 0.1 * q, 40)
        check(lib().amcafe_analytic_temp_curr(a.h, ctypes.byref(Laser(*at)), None))
        melted += b.temperature(*at)
    if easm:
        for d in (a, b):
            d.easm_temperature(100e-6, 100e-6, 40 * DX, 1.0, 0.0, 40, 200.0, 10e-6)
    f, g = a.download(), b.download()
    assert melted >= 12
    for k in f:
        assert np.array_equal(f[k], g[k]), k
