# SPDX-License-Identifier: MIT
"""The grid query against the oracle's pairs: crowds in which a body has as
many candidates as its segment of the pool holds (96 by default, 128 where the
pair pool is larger: what the group's memory holds), one less, one more and far
more, and a wide moving body above a multiple of the chunks of the large scan."""
import numpy as np
import pytest

import _oracle as O
import pmamd
import scenarios as S
from pmamd import layouts as L

pytestmark = pytest.mark.gpu


def crowd(n, seed, wide):
    """n small spheres in a ball of 0.6 m, flying side by side so fast that
    every proxy meets every other, far cubes of that width alone (they set the
    grid's cell), all in a random order, and with `wide` a dynamic slab."""
    rng = np.random.default_rng(seed)
    shapes = [("mesh", *S.box_mesh(50.0, 0.5, 50.0)), ("sphere", 0.01), ("mesh", *S.box_mesh(8.0, 0.1, 8.0)),
              ("mesh", *S.box_mesh(0.4, 0.4, 0.4))]
    way = rng.normal(size=(n, 3))
    near = 0.3 * way / np.linalg.norm(way, axis=1, keepdims=True) * rng.uniform(0.2, 1.0, (n, 1)) + (0, 12.0, 0)
    far = np.stack([4.0 * np.arange(40) - 80.0, np.full(40, 30.0), np.full(40, 5.0)], 1)
    order = rng.permutation(n + 40)
    body, fast = np.concatenate([near, far])[order], order < n
    pos = np.concatenate([[(0, -0.5, 0)], [(0, 6.0, 0)] if wide else np.zeros((0, 3)), body]).astype(np.float32)
    shape = np.concatenate([[0], [2] if wide else [], np.where(fast, 1, 3)]).astype(int)
    motion = np.full(len(pos), L.MOTION_DYNAMIC, np.uint32)
    motion[0] = L.MOTION_STATIC
    p = S.params(len(pos), motion=motion, mass=1.0, inertia=(0.1, 0.1, 0.1), shape=shape, margin=1e-4)
    st = S.states(len(pos), pos)
    st["linear_velocity"][len(pos) - n - 40:][fast] = 42.0
    return S.Scene(shapes, p, st)


@pytest.mark.parametrize("n", [2, 33, 64, 65, 96, 97, 98, 128, 129, 130, 170])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("pairs_per_body", [96, 192])
def test_crowds_give_the_oracles_pairs(n, wide, pairs_per_body):
    print("crowd", n, wide, pairs_per_body, flush=True)
    s = crowd(n, n, wide)
    g = s.build(pmamd.World(profile=1, pairs_per_body=pairs_per_body))
    o = s.build(O.OracleWorld(profile=1, lanes=32))
    g.step(1)
    o.step(1)
    want = o.pairs()
    assert len(want) >= n * (n - 1) // 2
    assert np.array_equal(g.pairs(), want)


@pytest.mark.parametrize("n", [1020, 1025, 2600])
def test_a_wide_body_meets_every_chunk(n):
    print("slab over", n, flush=True)
    rng = np.random.default_rng(n)
    shapes = [("mesh", *S.box_mesh(50.0, 0.5, 50.0)), ("sphere", 0.1), ("mesh", *S.box_mesh(40.0, 0.1, 40.0))]
    side = int(np.ceil(np.sqrt(n)))
    k = np.arange(n)
    pos = np.stack([1.4 * (k % side) - 0.7 * side, np.where(rng.random(n) < 0.5, 8.0, 60.0), 1.4 * (k // side) - 0.7 * side], 1)
    pos = np.concatenate([[(0, -0.5, 0), (0, 6.0, 0)], pos]).astype(np.float32)
    motion = np.full(n + 2, L.MOTION_DYNAMIC, np.uint32)
    motion[0] = L.MOTION_STATIC
    p = S.params(n + 2, motion=motion, mass=1.0, inertia=(0.1, 0.1, 0.1), shape=np.array([0, 2] + [1] * n), margin=1e-3)
    s = S.Scene(shapes, p, S.states(n + 2, pos))
    g = s.build(pmamd.World(profile=1))
    o = s.build(O.OracleWorld(profile=1, lanes=32))
    g.step(1)
    o.step(1)
    assert np.array_equal(g.pairs(), o.pairs())
