# SPDX-License-Identifier: MIT
"""The triangle-pair path against the oracle's serial one, bit for bit: shape
pairs from one leaf pair to 64 (all that a screened pair's mask holds) and
more, flying, resting and crossing, so that pairs leave at the screen, carry
their cells through it or pass it unseen, and candidates fill a batch in part,
exactly or several times."""
import numpy as np
import pytest

import _oracle as O
import pmamd
import scenarios as S
from pmamd import layouts as L
from test_gpu_face_rows import cone

pytestmark = pytest.mark.gpu


def wedge():
    """A non-convex closed mesh (an L-shaped prism): no planes."""
    o = [(0, 0), (0.4, 0), (0.4, 0.15), (0.15, 0.15), (0.15, 0.4), (0, 0.4)]
    v = [(x - 0.15, y - 0.15, z) for z in (-0.1, 0.1) for x, y in o]
    caps = [(0, 1, 2), (0, 2, 3), (0, 3, 4), (0, 4, 5)]
    idx = [k for c in caps for k in (c[0], c[2], c[1])] + [6 + k for c in caps for k in c]
    for k in range(6):
        a, b = k, (k + 1) % 6
        idx += [a, b, 6 + b, a, 6 + b, 6 + a]
    return np.array(v, np.float32), np.array(idx, np.uint32)


def scene(speed, seed):
    """Couples of bodies far from each other: near, touching or crossing."""
    rng = np.random.default_rng(seed)
    shapes = [("mesh", *S.box_mesh(8.0, 0.5, 8.0)), ("mesh", *S.box_mesh(0.2, 0.15, 0.25)), ("mesh", *wedge())]
    shapes += [("mesh", *cone(k)) for k in (3, 8, 15, 17, 18, 24)] + [("mesh", *S.cube_sphere_mesh(0.25))]
    kinds = [(i, j) for i in range(1, len(shapes)) for j in range(i, len(shapes))]
    pos, shape = [(0.0, -20.0, 0.0)], [0]
    for k, (i, j) in enumerate(kinds):
        c = np.array([2.0 * (k % 8), 2.0 * (k // 8), 0.0])
        way = rng.normal(size=3)
        way /= np.linalg.norm(way)
        d = rng.uniform(0.15, 0.45)
        pos += [c - way * d / 2, c + way * d / 2]
        shape += [i, j]
    n = len(pos)
    motion = np.full(n, L.MOTION_DYNAMIC, np.uint32)
    motion[0] = L.MOTION_STATIC
    p = S.params(n, motion=motion, mass=1.0, inertia=(0.02, 0.02, 0.02), shape=np.array(shape), margin=S.REF_MARGIN)
    st = S.states(n, np.array(pos, np.float32))
    q = rng.normal(size=(n, 4))
    q[0] = (0, 0, 0, 1)
    st["orientation"] = (q / np.linalg.norm(q, axis=1, keepdims=True)).astype(np.float32)
    st["linear_velocity"][1:] = rng.normal(0, speed, (n - 1, 3))
    st["angular_velocity"][1:] = rng.normal(0, speed, (n - 1, 3))
    return S.Scene(shapes, p, st)


@pytest.mark.parametrize("speed", [0.0, 2.0, 12.0])
@pytest.mark.parametrize("seed", [1, 2, 3])
def test_triangle_pairs_equal_the_serial_path(speed, seed):
    print("couples", speed, seed, flush=True)
    s = scene(speed, seed)
    g = s.build(pmamd.World(profile=0, base_iterations=2))
    o = s.build(O.OracleWorld(profile=0, base_iterations=2, lanes=32))
    for _ in range(2):
        g.step(1)
        o.step(1)
        assert np.array_equal(g.pairs(), o.pairs())
        for f in ("triangle_pairs", "fallback_pairs"):
            assert g.stats()[f] == o.stats()[f]
        gm, om = g.manifolds(), o.manifolds()
        assert np.array_equal(gm["count"], om["count"])
        live = np.arange(8)[None, :] < gm["count"][:, None]
        for f in ("normal", "point", "penetration", "impact_fraction", "persistent"):
            assert np.array_equal(gm["contacts"][f][live], om["contacts"][f][live]), f
        o.set_states(g.states())
        g.set_states(g.states())
