# SPDX-License-Identifier: MIT
"""The dataflow sweep's mailboxes are addressed with 32 bits: the rule that
keeps larger worlds off them, on the CPU, and the form of one launch per
colour that those worlds take against the sweep, bit for bit."""
import os
import subprocess

import numpy as np
import pytest

import pmamd
import scenarios as S
from test_build_checks import build, needs_hipcc
from test_gpu_joint_rows import hub

RULE = r"""
#include "pmh_internal.hpp"
#include <cstdio>
int main() {
    unsigned n;
    while (std::scanf("%u", &n) == 1)
        std::printf("%d %zu %u %u\n", pmh::flow_fits(n) ? 1 : 0, pmh::flow_words(n), pmh::flow_offset(n - 1), pmh::flow_offset(n));
    return 0;
}
"""


@needs_hipcc
def test_every_mailbox_of_the_sweep_is_within_reach(tmp_path):
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(RULE)
    subprocess.run([build.HIPCC, "-std=c++17", "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-I", build.SRC, "-I",
                    "/opt/rocm/include", str(src), "-o", str(exe)], check=True, capture_output=True)
    sizes = [1, 4096, 2 ** 25, 2 ** 26 - 1, 2 ** 26, 2 ** 26 + 1, 2 ** 27, 2 ** 30 - 1, 2 ** 32 - 1]
    out = subprocess.run([str(exe)], input="\n".join(map(str, sizes)), capture_output=True, text=True, check=True).stdout
    for n, line in zip(sizes, out.splitlines()):
        fits, words, last, end = map(int, line.split())
        assert fits == (64 * n < 2 ** 32), n
        assert words == (8 * n if fits else 0), n
        if fits:
            assert (last, end) == (64 * (n - 1), 64 * n), n


@pytest.mark.gpu
@pytest.mark.parametrize("lanes", [8, 16, 32, 64])
@pytest.mark.parametrize("profile", [0, 1])
@pytest.mark.parametrize("scene", ["pyramid", "hub"])
def test_one_launch_per_colour_equals_the_sweep(scene, lanes, profile):
    print("per colour", scene, lanes, profile, flush=True)
    s = S.pyramid(rows=9) if scene == "pyramid" else hub(33, profile)
    worlds = [s.build(pmamd.World(profile=profile, base_iterations=6, solve_lanes=lanes, per_color_sweep=per))
              for per in (False, True)]
    for _ in range(3):
        for w in worlds:
            w.step(1)
        a, b = (w.states() for w in worlds)
        for f in ("position", "orientation", "linear_velocity", "angular_velocity"):
            np.testing.assert_array_equal(a[f], b[f], err_msg=f)
        a, b = (w.manifolds() for w in worlds)
        live = np.arange(8)[None, :] < a["count"][:, None]
        np.testing.assert_array_equal(a["count"], b["count"])
        for f in ("avbd_dual", "accumulated_normal_impulse", "avbd_anchor_a"):
            np.testing.assert_array_equal(a["contacts"][f][live], b["contacts"][f][live], err_msg=f)
    if scene == "hub":
        for f in ("rows", "applied_impulse", "broken"):
            assert worlds[0].joints()[f].tobytes() == worlds[1].joints()[f].tobytes(), f
