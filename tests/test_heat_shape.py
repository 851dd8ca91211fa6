"""The heat field's launch shape over the whole range of `checkpoint` (the steps of a launch, any
positive int) and over domains down to one voxel: a host computation, so no GPU is needed.  A segment is no
longer than the call; the shares of every launch cover its column tiles once, none of them with more
than its part; and the block slots stay within the allocation-free call's array."""
import ctypes
import itertools

import pytest

import amcafe_amd
from amcafe_amd.heat import track_desc

DOMAINS = [(1, 1, 1), (64, 1, 4), (128, 1, 1), (1, 40, 30), (1, 129, 1), (2, 17, 9), (64, 32, 16), (125, 99, 41),
           (256, 256, 64), (2 ** 31 - 1, 1, 1), (1, 2 ** 31 - 1, 1), (1 << 20, 1, 2047)]
CHECKPOINTS = [0, 1, 2, 7, 100, 2000, 100000, 2 ** 20 + 1, 2 ** 25, 2 ** 30, 2 ** 31 - 1]
STEPS = [0, 1, 20, 100, 200, 2 ** 31 - 1]


def _shape(d, nsteps, fp64, steps):
    o = (ctypes.c_int * 5)()
    amcafe_amd.lib().amcd_heat_shape(ctypes.byref(d), nsteps, fp64, steps, o)
    return list(o)


@pytest.mark.parametrize("fp64", [0, 1])
@pytest.mark.parametrize("nX", DOMAINS)
def test_shares_cover_every_launch(nX, fp64):
    blocks = (nX[0] * nX[1] * nX[2] + 255) // 256
    for checkpoint, nsteps in itertools.product(CHECKPOINTS, STEPS):
        d = track_desc(nX, steps=10, checkpoint=checkpoint)
        groups, runs, seg, _, ct = _shape(d, nsteps, fp64, 0)
        want = min(checkpoint or 100, max(nsteps, 1))
        assert 1 <= seg <= want, (checkpoint, nsteps, seg)
        assert seg == want or (seg + 1) * nX[0] > 1 << 30, (checkpoint, nsteps, seg)
        assert groups >= 1 and 1 <= runs <= 65535
        # rows in groups of 128, lines or patches padded to at most 1.9 times
        assert groups * 128 >= nX[1] * nX[2] and groups <= 1.9 * nX[1] * nX[2] / 128 + 1
        assert groups * runs <= 2 * blocks, (checkpoint, nsteps, groups, runs)
        for steps in {min(seg, nsteps), nsteps % seg, 0}:
            tiles = (steps * nX[0] + ct - 1) // ct
            ctiles = _shape(d, nsteps, fp64, steps)[3]
            assert ctiles == -(-tiles // runs), (checkpoint, nsteps, steps, runs, ctiles)
            assert ctiles * runs < 2 ** 31


def test_a_long_checkpoint_is_the_calls_length():
    d, e = track_desc((125, 99, 41), steps=200, checkpoint=200), track_desc((125, 99, 41), steps=200, checkpoint=10 ** 6)
    for fp64 in (0, 1):
        assert _shape(d, 200, fp64, 200) == _shape(e, 200, fp64, 200)
