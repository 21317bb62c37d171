# SPDX-License-Identifier: MIT
"""Islands of known shape: rows of boxes in contact end to end on a static
floor, the bodies in random order.  Every row is one island, and each of its
bodies' parent is the row's smallest index, on every step (the trees behind it
are as deep as they get: a row is a path)."""
import numpy as np
import pytest

import pmamd
import scenarios as S
from pmamd import layouts as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,length", [(3, 5), (1, 250), (40, 90), (9000, 1), (30, 400), (60, 500)])
def test_every_body_points_at_the_smallest_index_of_its_row(rows, length):
    print("rows", rows, length, flush=True)
    n = rows * length
    rng = np.random.default_rng(rows)
    order = rng.permutation(n)
    row = np.arange(n) // length
    pos = np.stack([(np.arange(n) % length) * 0.3005, np.full(n, 0.1502), row * 1.5], 1)[order]
    row = row[order]
    shapes = [("mesh", *S.box_mesh(0.15 * length + 5.0, 0.5, 0.75 * rows + 5.0)), ("mesh", *S.box_mesh(0.15, 0.15, 0.15))]
    centre = np.array([0.15 * length, 0.0, 0.75 * rows])
    motion = np.full(n + 1, L.MOTION_DYNAMIC, np.uint32)
    motion[0] = L.MOTION_STATIC
    p = S.params(n + 1, motion=motion, mass=10.0, inertia=S.box_inertia(10.0, (0.15, 0.15, 0.15)),
                 shape=np.minimum(np.arange(n + 1), 1), margin=S.REF_MARGIN)
    st = S.states(n + 1, np.concatenate([[centre - [0.0, 0.5, 0.0]], pos]).astype(np.float32))
    w = S.Scene(shapes, p, st).build(pmamd.World(profile=0, base_iterations=2, pairs_per_body=32, points_per_body=32))
    first = np.full(rows, n + 1, np.int64)
    np.minimum.at(first, row, np.arange(1, n + 1))
    for _ in range(4):
        w.step(1)
        b = w.bodies()
        assert np.array_equal(b["parent"][1:], first[row])
        assert w.stats()["islands"] == rows
        # the impact flag is the island's
        flag = np.zeros(rows, np.int64)
        np.maximum.at(flag, row, b["impact"][1:])
        assert np.array_equal(b["impact"][1:], flag[row])
