# SPDX-License-Identifier: MIT
"""Mesh pairs whose leaf pairs do not fit in a wavefront's list: evaluated in
order by the serial functions on four lanes, one of which writes the manifold.
Two fine sheets on each other overlap in more than 512 leaf pairs: a
world of at most eight bodies allows 4096 candidates, a larger one sends them
down the traversal, whose list they outgrow too.  Bit for bit against the
oracle."""
import numpy as np
import pytest

import _oracle as O
import pmamd
import scenarios as S
from pmamd import layouts as L

pytestmark = pytest.mark.gpu


def sheet(cells, size, wave):
    """An open sheet of cells x cells squares, its heights a wave."""
    g = np.linspace(-size, size, cells + 1)
    x, z = np.meshgrid(g, g, indexing="ij")
    v = np.stack([x, wave * np.sin(9 * x) * np.cos(7 * z), z], -1).reshape(-1, 3)
    idx = []
    for i in range(cells):
        for j in range(cells):
            k = i * (cells + 1) + j
            idx += [k, k + 1, k + cells + 1, k + 1, k + cells + 2, k + cells + 1]
    return v.astype(np.float32), np.array(idx, np.uint32)


def scene(bodies, apart, speed, wave):
    shapes = [("mesh", *S.box_mesh(8.0, 0.5, 8.0)), ("mesh", *sheet(20, 0.3, wave)), ("mesh", *S.cube_sphere_mesh(0.1))]
    motion = np.full(bodies, L.MOTION_DYNAMIC, np.uint32)
    motion[0] = L.MOTION_STATIC
    shape = np.full(bodies, 2)
    shape[:3] = (0, 1, 1)
    pos = np.zeros((bodies, 3), np.float32)
    pos[:, 0] = 3.0 + 1.0 * np.arange(bodies)
    pos[0] = (0, -20, 0)
    pos[1] = (0, 0, 0)
    pos[2] = (0.02, apart, 0.01)
    p = S.params(bodies, motion=motion, mass=1.0, inertia=(0.04, 0.04, 0.04), shape=shape, margin=S.REF_MARGIN)
    st = S.states(bodies, pos)
    st["orientation"][2] = S.quat((0, 1, 0), 0.4)
    st["linear_velocity"][1] = (0, speed, 0)
    st["angular_velocity"][2] = (0, speed, 0)
    return S.Scene(shapes, p, st)


@pytest.mark.parametrize("bodies,fallback", [(8, 0), (9, 1)])
@pytest.mark.parametrize("apart,speed,wave", [(0.001, 0.0, 0.0), (0.004, 0.0, 0.02), (0.03, 1.0, 0.02), (0.08, 6.0, 0.02)])
def test_pairs_that_outgrow_the_list_equal_the_serial_path(bodies, fallback, apart, speed, wave):
    print("sheets", bodies, apart, speed, wave, flush=True)
    s = scene(bodies, apart, speed, wave)
    g = s.build(pmamd.World(profile=0, base_iterations=2))
    o = s.build(O.OracleWorld(profile=0, base_iterations=2, lanes=32))
    for step in range(2):
        g.step(1)
        o.step(1)
        assert np.array_equal(g.pairs(), o.pairs())
        for f in ("triangle_pairs", "fallback_pairs"):
            assert g.stats()[f] == o.stats()[f]
        if step == 0:   # more than 512 leaf pairs, and at most 4096
            assert (o.stats()["triangle_pairs"], o.stats()["fallback_pairs"]) == (1, fallback)
        gm, om = g.manifolds(), o.manifolds()
        assert np.array_equal(gm["count"], om["count"])
        assert om["count"].max() > 0
        live = np.arange(8)[None, :] < gm["count"][:, None]
        for f in ("normal", "point", "penetration", "impact_fraction"):
            assert np.array_equal(gm["contacts"][f][live], om["contacts"][f][live]), f
        o.set_states(g.states())
        g.set_states(g.states())
