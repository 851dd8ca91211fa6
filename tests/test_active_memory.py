"""Device memory per active cell: every domain holds an eighth of its voxels (at least 65,536) in capacity, so
it bounds how many domains a batch can have on a card.  2,211 bytes a cell is what the arrays took as
one per field; a record for every candidate of every active cell took 3,309."""
import ctypes

import pytest

import amcafe_amd


@pytest.mark.parametrize("cells", [1, 63, 64, 1000, 65536, 4194304, 1 << 23, 70_000_000, 90_000_000])
def test_bytes_per_active_cell(cells):
    f = amcafe_amd.lib().amcd_active_bytes
    f.restype, f.argtypes = ctypes.c_size_t, [ctypes.c_int]
    assert f(cells) <= 2211 * cells + 20 * 512  # (every array is padded)
