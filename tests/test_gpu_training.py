# SPDX-License-Identifier: MIT
"""The training kernel, one update at a time, against Adam in float64 on the
gradients that the gradient kernel gives at the same parameters: the first
k epochs of a run are the same whatever its length, so the parameters after
k - 1 epochs are where update k starts, bit for bit.

Sizes: one sample, both sides of a full 16-sample tile and of a full
minibatch, and minibatches with a ragged last one."""
import numpy as np
import pytest

import pmamd

pytestmark = pytest.mark.gpu

LR = 1e-2


def permutations(seed, n, epochs):
    state, mask, out = (seed * 747796405 + 2891336453) & 0xFFFFFFFF, 0xFFFFFFFF, []
    for _ in range(epochs):
        o = list(range(n))
        for k in range(n - 1, 0, -1):
            state = (state * 1664525 + 1013904223) & mask
            j = (state * (k + 1)) >> 32
            o[k], o[j] = o[j], o[k]
        out.append(np.array(o))
    return out


def samples_of(n):
    rng = np.random.default_rng(n)
    return rng.normal(0, 1, (n, 18)).astype(np.float32)


class Adam:
    def __init__(self):
        self.m = np.zeros(pmamd.MLP_PARAMS)
        self.v = np.zeros(pmamd.MLP_PARAMS)
        self.t = 0

    def step(self, p, g):
        g = g.astype(np.float64)
        self.t += 1
        self.m = 0.9 * self.m + 0.1 * g
        self.v = 0.999 * self.v + 0.001 * g * g
        mh, vh = self.m / (1 - 0.9 ** self.t), self.v / (1 - 0.999 ** self.t)
        return p - LR * mh / (np.sqrt(vh) + 1e-8)


@pytest.mark.parametrize("n", (1, 15, 16, 17, 63, 64))
def test_each_update_of_a_single_minibatch(n):
    s, epochs = samples_of(n), 4
    order, adam, p = permutations(11, n, epochs), Adam(), pmamd.warmstart_init(5)
    live = pmamd.MLP_PARAMS - 2                       # then the bounds, the targets' maxima
    for k in range(epochs):
        loss, g = pmamd.warmstart_gradients(p, s[order[k]])
        want = adam.step(p.astype(np.float64), g)
        q, losses = pmamd.warmstart_train(s, epochs=k + 1, learning_rate=LR, seed=11, params=pmamd.warmstart_init(5))
        # float32 Adam: 1 - 0.999^t is 1 - 0.999f^t with the constant's
        # rounding (2^-25 of 0.999, amplified by 1 / (1 - 0.999) = 1000 in the
        # correction, halved by the root: 1.5e-5 of a step), a dozen roundings
        # of 2^-24 of a step; the new parameter's own rounding.  A step is at
        # most 1 / sqrt(1 - 0.999) of the rate.
        bound = 3e-5 * np.abs(want - p) + 2.0 ** -23 * np.abs(want) + 1e-6 * LR
        assert (np.abs(q[:live] - want[:live]) <= bound[:live]).all(), k
        assert np.array_equal(q[live:], np.maximum(s[:, 16:].max(axis=0), 0.0))
        assert abs(losses[k] - loss) <= 1e-6 * loss      # the same sums
        p = q


@pytest.mark.parametrize("n", (65, 128, 200))
def test_epochs_of_several_minibatches(n):
    s, epochs = samples_of(n), 2
    order, adam, p = permutations(11, n, epochs), Adam(), pmamd.warmstart_init(5).astype(np.float64)
    live, steps = pmamd.MLP_PARAMS - 2, 0
    for o in order:
        for first in range(0, n, 64):
            _, g = pmamd.warmstart_gradients(p.astype(np.float32), s[o[first:first + 64]])
            p, steps = adam.step(p, g), steps + 1
    q, _ = pmamd.warmstart_train(s, epochs=epochs, learning_rate=LR, seed=11, params=pmamd.warmstart_init(5))
    # Between updates a parameter next to a bf16 rounding boundary may round
    # the other way on one side: a weight off by 2^-8 moves the gradients by
    # at most about that, and so the steps.
    assert np.abs(q[:live] - p[:live]).mean() <= 2.0 ** -8 * LR * steps
