# SPDX-License-Identifier: MIT
"""Worlds whose scans end on and next to a tile, a whole short scan and the
sizes from which the totals are scanned by their own launch: couples of cubes
in contact, so that pairs, points and the contact cache (each placed by a
scan) fill exactly, two steps against the oracle."""
import numpy as np
import pytest

import _oracle as O
import pmamd
import scenarios as S
from pmamd import layouts as L

pytestmark = pytest.mark.gpu


def couples(n):
    """n bodies: a static cube, then couples one above the other, apart."""
    k = np.arange(n - 1)
    side = int(np.ceil(np.sqrt(n / 2)))
    pos = np.zeros((n, 3), np.float32)
    pos[0] = (-5.0, 0.0, -5.0)
    pos[1:, 0] = 1.5 * (k // 2 % side)
    pos[1:, 1] = 0.3995 * (k % 2)
    pos[1:, 2] = 1.5 * (k // 2 // side)
    motion = np.full(n, L.MOTION_DYNAMIC, np.uint32)
    motion[0] = L.MOTION_STATIC
    p = S.params(n, motion=motion, mass=1.0, inertia=S.box_inertia(1.0, (0.2, 0.2, 0.2)), shape=np.zeros(n, int),
                 margin=S.REF_MARGIN)
    return S.Scene([("mesh", *S.box_mesh(0.2, 0.2, 0.2))], p, S.states(n, pos))


# 8192 elements are the longest short scan; 44000 bodies have more than 4096
# tiles of pair slots.
@pytest.mark.parametrize("n", [5, 1023, 1024, 1025, 4096, 4097, 8191, 8192, 8193, 9216, 44000])
def test_scans_of_every_length(n):
    print("couples", n, flush=True)
    s = couples(n)
    g = s.build(pmamd.World(profile=1))
    o = s.build(O.OracleWorld(profile=1, lanes=32))
    for _ in range(2):
        g.step(1)
        o.step(1)
    assert np.array_equal(g.pairs(), o.pairs()) and len(g.pairs()) >= (n - 1) // 2
    gs, os_ = g.stats(), o.stats()
    for f in ("manifolds", "points", "cache_hits"):
        assert gs[f] == os_[f], f
    a, b = g.states(), o.states()
    for f in ("position", "orientation", "linear_velocity", "angular_velocity"):
        np.testing.assert_array_equal(a[f], b[f], err_msg=f)
