# SPDX-License-Identifier: MIT
"""Clipped polygons that outgrow a row of lanes in worlds where none is expected
to (shapes of at most 13 triangles): the row's limit is lowered, so that some of
them or all do, and every manifold of every step is the oracle's."""
import numpy as np
import pytest

import _oracle as O
import pmamd
import scenarios as S
from test_gpu_face_rows import scene as cones

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limit", [0, 3, 4, 5, 6, 16])
@pytest.mark.parametrize("kind", ["pyramid", "resting cones", "falling cones"])
def test_polygons_wider_than_the_row_go_on_on_one_lane(kind, limit):
    print("wide", kind, limit, flush=True)
    s = S.pyramid(rows=6) if kind == "pyramid" else cones(7, -0.004 if kind == "resting cones" else 0.02,
                                                          1.0 if kind == "resting cones" else 30.0)
    g = s.build(pmamd.World(profile=0, base_iterations=4))
    o = s.build(O.OracleWorld(profile=0, base_iterations=4, lanes=32))
    g.set_face_row_limit(limit)
    for _ in range(4):   # pairs leave and move up the list between steps
        g.step(1)
        o.step(1)
        assert np.array_equal(g.pairs(), o.pairs())
        gm, om = g.manifolds(), o.manifolds()
        assert om["count"].max() > 0
        assert np.array_equal(gm["count"], om["count"])
        assert np.array_equal(gm["face_patch"], om["face_patch"])
        live = np.arange(8)[None, :] < gm["count"][:, None]
        for f in ("normal", "point", "penetration", "impact_fraction", "persistent"):
            assert np.array_equal(gm["contacts"][f][live], om["contacts"][f][live]), f
        o.set_states(g.states())
        g.set_states(g.states())
