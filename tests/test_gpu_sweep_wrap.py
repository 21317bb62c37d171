# SPDX-License-Identifier: MIT
"""Sweeps are numbered with 32 bits: a step across the wrap of the number
solves every iteration and equals one far from it, bit for bit, wherever in the
step the wrap falls."""
import numpy as np
import pytest

import pmamd
import scenarios as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("before", range(0, 10, 2))
@pytest.mark.parametrize("profile", [0, 1])
def test_a_step_across_the_wrap(before, profile):
    print("wrap", before, profile, flush=True)
    scene = S.pyramid(rows=5)
    worlds = [scene.build(pmamd.World(profile=profile, base_iterations=4)) for _ in range(2)]
    # The stamp so far is even: the realtime profile makes 8 sweeps a step,
    # the other 4 or 8.
    for w in worlds:
        w.step(2)
    worlds[1].set_sweep_stamp(2 ** 32 - 2 - before)
    for _ in range(3):
        for w in worlds:
            w.step(1)
        a, b = (w.states() for w in worlds)
        for f in ("position", "orientation", "linear_velocity", "angular_velocity"):
            np.testing.assert_array_equal(a[f], b[f], err_msg=f)
