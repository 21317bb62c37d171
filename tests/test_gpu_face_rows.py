# SPDX-License-Identifier: MIT
"""The convex face path on rows of lanes against the oracle's serial one, bit
for bit: reference faces with few and many side planes (a polygon clipped by
17 of them has more vertices than a row has lanes), bodies that touch at the
end of a step, at its start, at a time in between, or not at all."""
import numpy as np
import pytest

import _oracle as O
import pmamd
import scenarios as S
from pmamd import layouts as L

pytestmark = pytest.mark.gpu


def cone(sides, radius=0.3, height=0.5):
    """A convex cone: `sides` triangles around, sides - 2 in the base."""
    a = 2 * np.pi * np.arange(sides) / sides
    v = np.concatenate([np.stack([radius * np.cos(a), np.full(sides, -height / 4), radius * np.sin(a)], 1),
                        [[0.0, 0.75 * height, 0.0]]]).astype(np.float32)
    idx = []
    for k in range(sides):
        idx += [k, sides, (k + 1) % sides]
    for k in range(1, sides - 1):
        idx += [0, k, k + 1]
    return v, np.array(idx, np.uint32)


def scene(sides, gap, speed):
    """A floor, wide dynamic boxes on it and a cone over each: on one triangle
    of the box's top, across its diagonal, over an edge, and tilted."""
    shapes = [("mesh", *S.box_mesh(8.0, 0.5, 8.0)), ("mesh", *S.box_mesh(1.0, 0.25, 1.0)), ("mesh", *cone(sides))]
    spots = [(0.45, -0.45, 0.0), (0.0, 0.05, 0.0), (0.95, 0.1, 0.0), (-0.3, 0.4, 0.06)]
    pos, shape, rot = [(0.0, -0.5, 0.0)], [0], [(0, 0, 0, 1)]
    for k in range(4):
        pos.append((3.0 * k - 4.5, 0.2495, 0.0))
        shape.append(1)
        rot.append((0, 0, 0, 1))
    for k, (x, z, tilt) in enumerate(spots):
        pos.append((3.0 * k - 4.5 + x, 0.4995 + 0.125 + gap, z))
        shape.append(2)
        rot.append(S.quat((1, 0, 1), tilt))
    n = len(pos)
    motion = np.full(n, L.MOTION_DYNAMIC, np.uint32)
    motion[0] = L.MOTION_STATIC
    p = S.params(n, motion=motion, mass=2.0, inertia=(0.2, 0.2, 0.2), shape=np.array(shape), margin=S.REF_MARGIN)
    st = S.states(n, np.array(pos, np.float32))
    st["orientation"] = np.array(rot, np.float32)
    st["linear_velocity"][5:, 1] = -speed
    return S.Scene(shapes, p, st)


@pytest.mark.parametrize("sides", [3, 4, 7, 8, 9, 12, 15, 16, 17])
@pytest.mark.parametrize("gap,speed", [(5e-4, 0.0), (-0.004, 1.0), (0.05, 6.0), (0.02, 30.0), (0.4, 1.0)])
def test_face_rows_equal_the_serial_path(sides, gap, speed):
    print("cone", sides, gap, speed, flush=True)
    s = scene(sides, gap, speed)
    g = s.build(pmamd.World(profile=0, base_iterations=2))
    o = s.build(O.OracleWorld(profile=0, base_iterations=2, lanes=32))
    for _ in range(2):
        g.step(1)
        o.step(1)
        assert np.array_equal(g.pairs(), o.pairs())
        gm, om = g.manifolds(), o.manifolds()
        assert np.array_equal(gm["count"], om["count"])
        assert np.array_equal(gm["face_patch"], om["face_patch"])
        live = np.arange(8)[None, :] < gm["count"][:, None]
        for f in ("normal", "point", "penetration", "impact_fraction", "persistent"):
            assert np.array_equal(gm["contacts"][f][live], om["contacts"][f][live]), f
        o.set_states(g.states())
        g.set_states(g.states())
