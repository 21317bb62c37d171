# SPDX-License-Identifier: MIT
"""The dataflow sweep's lane forms against the oracle in the same summation
order: bodies with fewer and with more contact points than lanes, a wavefront
whose last bodies are padding, and a block that only the equilibrated second
attempt of the solve can factor."""
import numpy as np
import pytest

import _oracle as O
import pmamd
import scenarios as S
from pmamd import layouts as L

pytestmark = pytest.mark.gpu


def star(arms, ratio=1.0):
    """One box on a floor with `arms` boxes resting on it: 4 arms + 4 points
    on the middle body (records for the kernel seam), its mass `ratio` times
    theirs."""
    n = arms + 2
    motion = np.full(n, L.MOTION_DYNAMIC, np.uint32)
    motion[0] = L.MOTION_STATIC
    mass = np.ones(n, np.float32)
    mass[1] = ratio
    p = S.params(n, motion=motion, mass=mass, inertia=mass[:, None] * np.float32([0.1, 0.1, 0.1]), margin=0.005)
    pos = np.zeros((n, 3), np.float32)
    pos[1] = (0, 0.5, 0)
    pos[2:, 0] = np.linspace(-0.4, 0.4, arms)
    pos[2:, 1] = 1.25
    prev = S.states(n, pos)
    cur = prev.copy()
    cur["linear_velocity"][1:, 1] = np.float32(-9.81) * S.DT
    cur["position"][1:] += cur["linear_velocity"][1:] * S.DT
    pairs = np.array([n] + [k * n + 1 for k in range(2, n)], np.uint32)
    m = np.zeros(len(pairs), L.MANIFOLD)
    m["count"] = 4
    rng = np.random.default_rng(arms)
    for k in range(len(pairs)):
        x = 0.0 if k == 0 else pos[k + 1, 0]
        y = 0.0 if k == 0 else 1.0
        m[k]["contacts"]["normal"][:4] = (0, 1, 0)
        m[k]["contacts"]["point"][:4] = [(x + dx, y, dz) for dx in (-0.05, 0.05) for dz in (-0.2, 0.2)]
        m[k]["contacts"]["penetration"][:4] = rng.uniform(-2e-4, 2e-3, 4)
    return p, prev, cur, m, pairs


@pytest.mark.parametrize("arms", [1, 6, 7, 8, 15, 16, 40])
@pytest.mark.parametrize("ratio", [1.0, 1.0e-6, 1.0e6])
@pytest.mark.parametrize("profile", [0, 1])
def test_points_around_the_lane_count(arms, ratio, profile):
    print("star", arms, ratio, profile, flush=True)
    p, prev, cur, m, pairs = star(arms, ratio)
    outs = []
    for solve in (pmamd.prepare_solve, lambda *a, **k: O.prepare_solve(*a, lanes=32, **k)):
        c, mm, b = cur.copy(), m.copy(), np.zeros(len(p), L.AVBD_BODY)
        solve(p, prev, c, mm, pairs, bodies=b, profile=profile)
        outs.append((c, mm))
    # the same operations in the same order: equal bits
    for f in ("position", "orientation", "linear_velocity", "angular_velocity"):
        np.testing.assert_array_equal(outs[0][0][f], outs[1][0][f])
    for f in ("avbd_dual", "accumulated_normal_impulse", "avbd_anchor_a"):
        np.testing.assert_array_equal(outs[0][1]["contacts"][f], outs[1][1]["contacts"][f])


@pytest.mark.parametrize("lanes", [8, 16, 32, 64])
@pytest.mark.parametrize("rows", [3, 9])
def test_every_lane_setting_follows_the_oracle(lanes, rows):
    print("pyramid", lanes, rows, flush=True)
    scene = S.pyramid(rows=rows)
    g = scene.build(pmamd.World(profile=0, base_iterations=6, solve_lanes=lanes))
    o = scene.build(O.OracleWorld(profile=0, base_iterations=6, lanes=lanes))
    g.step(4)
    o.step(4)
    assert np.array_equal(g.pairs(), o.pairs())
    gs, os_ = g.states(), o.states()
    # equal operations; only atan2f in large rotations may differ by an ulp
    for f in ("position", "linear_velocity", "orientation", "angular_velocity"):
        np.testing.assert_allclose(gs[f], os_[f], rtol=1e-5, atol=1e-5)
