# SPDX-License-Identifier: MIT
"""A sweep wait that runs out is never passed over: with a short wait limit a
step either fails and keeps its states, or every word it took had arrived and
its result is that of the default limit, bit for bit.  Boxes that slide, so
that the last update also takes the other end's rotation delta."""
import numpy as np
import pytest

import pmamd
import scenarios as S

pytestmark = pytest.mark.gpu
FIELDS = ("position", "orientation", "linear_velocity", "angular_velocity")


def sliding(rows):
    scene = S.pyramid(rows=rows)
    v = scene.states["linear_velocity"]
    v[1:, 0] = np.linspace(-1.0, 1.0, len(v) - 1)
    return scene


@pytest.mark.parametrize("lanes", [8, 32])
@pytest.mark.parametrize("rows", [2, 6])
@pytest.mark.parametrize("limit", [0, 20, 40, 80, 160])
def test_a_step_with_little_patience_fails_or_is_right(limit, rows, lanes):
    print("limit", limit, rows, lanes, flush=True)
    scene = sliding(rows)
    outcomes = []
    for steps in range(1, 9):
        reference = scene.build(pmamd.World(profile=0, base_iterations=4, solve_lanes=lanes))
        world = scene.build(pmamd.World(profile=0, base_iterations=4, solve_lanes=lanes))
        reference.step(steps)
        world.step(steps)
        world.set_sweep_wait_limit(limit)
        try:
            world.step(1)
            reference.step(1)
            outcomes.append("done")
        except pmamd.PmhError as e:
            assert e.code == -2
            outcomes.append("failed")
        a, b = world.states(), reference.states()
        for f in FIELDS:
            np.testing.assert_array_equal(a[f], b[f], err_msg=f"{f} after {steps} steps: {outcomes[-1]}")
        world.close()
        reference.close()
    print(outcomes, flush=True)
