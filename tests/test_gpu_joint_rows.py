# SPDX-License-Identifier: MIT
"""Joint rows against the oracle: a heavy hub with joints of every type and
option on it, as many as fall below, on and above the lanes of a group and
the 64 of a wavefront's list, some of them disabled and some breaking in the
step, so that the dealing of a body's joints over its lanes, the walk over
each joint's listed rows and both phases run."""
import numpy as np
import pytest

import _oracle as O
import pmamd
import scenarios as S
from pmamd import layouts as L

pytestmark = pytest.mark.gpu


def hub(arms, profile):
    """The hub falls onto a floor, its arms (spheres) around it in the air.
    Every fourth arm is the joint's first body."""
    n = arms + 2
    rng = np.random.default_rng(arms + 100 * profile)
    shapes = [("mesh",) + S.box_mesh(8.0, 0.5, 8.0), ("mesh",) + S.box_mesh(0.5, 0.5, 0.5), ("sphere", 0.05)]
    motion = np.full(n, L.MOTION_DYNAMIC, np.uint32)
    motion[0] = L.MOTION_STATIC
    shape = np.full(n, 2)
    shape[:2] = (0, 1)
    mass = np.full(n, 0.5, np.float32)
    mass[1] = 20.0
    inertia = np.full((n, 3), 0.01, np.float32)
    inertia[1] = S.box_inertia(20.0, (0.5, 0.5, 0.5))
    p = S.params(n, motion=motion, mass=mass, inertia=inertia, shape=shape, margin=0.005)
    pos = np.zeros((n, 3), np.float32)
    pos[0] = (0, -0.5, 0)
    pos[1] = (0, 0.51, 0)
    angle = 2.4 * np.arange(arms)
    pos[2:] = np.stack([1.4 * np.cos(angle), 1.0 + 0.12 * np.arange(arms), 1.4 * np.sin(angle)], axis=1)
    st = S.states(n, pos)
    st["linear_velocity"][1] = (0, -3.0, 0)
    st["angular_velocity"][1:] = rng.normal(0, 1.0, (n - 1, 3))
    joints = []
    zero = np.zeros((), L.JOINT_OPTIONS)
    for k in range(arms):
        kind = k % 8
        b = k + 2
        at_hub, at_arm = (pos[b] - pos[1]) * 0.9, -(pos[b] - pos[1]) * 0.1
        swap = k % 4 == 3
        o = L.joint_options(1, kind, b if swap else 1, 1 if swap else b, anchor_a=at_arm if swap else at_hub,
                            anchor_b=at_hub if swap else at_arm)
        o["local_orientation_a"] = S.quat((1, 0, 1), 0.03 * (k % 5))
        o["local_orientation_b"] = S.quat((0, 1, 0), 0.02 * (k % 7))
        for name in ("linear_limits", "angular_limits"):
            lim = zero[name].copy()
            lim["axes"] = (1 + k // 8) & 7
            lim["lower"] = (-0.02, -0.01, 0.0) if k % 3 else (0.01, 0.01, 0.01)
            lim["upper"] = (0.02, 0.03, 0.0) if k % 3 else (0.01, 0.05, 0.01)
            o[name] = lim
        for name in ("linear_springs", "angular_springs"):
            spr = zero[name].copy()
            spr["axes"] = (7 - k // 8) & 7
            spr["stiffness"] = (200.0, 100.0, 50.0)
            spr["damping"] = (2.0, 1.0, 0.5)
            o[name] = spr
        mot = zero["motor"].copy()
        mot["linear_enabled"], mot["angular_enabled"] = (k // 8) & 1, 1 - ((k // 16) & 1)
        mot["linear_target_velocity"], mot["linear_maximum_impulse"] = 0.5, 0.05
        mot["angular_target_velocity"], mot["angular_maximum_impulse"] = 3.0, 0.02
        o["motor"] = mot
        if k % 11 == 5:
            o["enabled"] = 0
        if k % 7 == 6:
            o["breaking_impulse_threshold"] = 0.05
        joints.append(o)
    return S.Scene(shapes, p, st, "hub", np.concatenate(joints))


@pytest.mark.parametrize("arms", [2, 7, 8, 9, 17, 32, 33, 65, 72])
@pytest.mark.parametrize("lanes,profile", [(8, 0), (32, 0), (64, 1), (16, 1)])
def test_a_hub_of_joints_follows_the_oracle(arms, lanes, profile):
    print("hub", arms, lanes, profile, flush=True)
    scene = hub(arms, profile)
    g = scene.build(pmamd.World(profile=profile, base_iterations=6, solve_lanes=lanes))
    o = scene.build(O.OracleWorld(profile=profile, base_iterations=6, lanes=lanes))
    for _ in range(2):
        g.step(1)
        o.step(1)
    gj, oj = g.joints(), o.joints()
    for f in ("enabled", "broken", "avbd_count", "avbd_next_a", "avbd_next_b"):
        np.testing.assert_array_equal(gj[f], oj[f], err_msg=f)
    gb, ob = g.bodies(), o.bodies()
    for f in ("color", "parent", "impact", "joint_head"):
        np.testing.assert_array_equal(gb[f], ob[f], err_msg=f)
    # equal operations in equal order; atan2f, sinf and cosf may differ by an
    # ulp, which two steps carry into the states and rows at this size
    gs, os_ = g.states(), o.states()
    for f in ("position", "orientation", "linear_velocity", "angular_velocity"):
        np.testing.assert_allclose(gs[f], os_[f], rtol=1e-4, atol=1e-4, err_msg=f)
    valid = np.arange(18)[None, :] < oj["avbd_count"][:, None]
    for f in ("error", "a", "b"):
        np.testing.assert_allclose(gj["rows"][f][valid], oj["rows"][f][valid], rtol=1e-4, atol=1e-4, err_msg=f)
