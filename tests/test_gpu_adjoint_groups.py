"""The differentiable form at the edges of its work split: 16 lanes per particle
up to 81,920 particles and 8 above, and a wave per particle from 1,025 candidates
on.  Forward bit for bit, gradients to the bound of test_gpu_adjoint (1e-9 of the
FP64 adjoint on the same recorded values, normwise)."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from tests.adjoint_cases import linear_loss_weights
from tests.test_gpu_adjoint import TOL, _compare, _cpu_grad, _gpu_grad

pytestmark = pytest.mark.gpu


def _check(tag, sc, steps):
    print(f"adjoint {tag}: n={sc.n}", flush=True)
    g = _gpu_grad(sc, steps, 1, lambda xs, ident: linear_loss_weights(xs.shape[0]))
    c = _cpu_grad(sc, steps, g["wx"], g["wv"])
    assert np.array_equal(g["x"].view(np.uint32), c["x"].view(np.uint32))
    assert np.array_equal(g["v"].view(np.uint32), c["v"].view(np.uint32))
    for k, e in _compare(tag, g, c).items():
        assert e < TOL, (tag, k, e)


@pytest.mark.parametrize("layers", [40, 41])
def test_lane_rule(layers):
    sc = scenes.small_dam(64, layers, 32, iters=2, seed=4)
    assert (sc.n <= 81920) == (layers == 40)
    _check(f"layers {layers}", sc, 1)


@pytest.mark.parametrize("pile", [1, 17, 1023, 1024, 1025, 1100])
def test_wave_rule(pile):
    h = 0.1
    base = scenes.small_dam(6, 5, 4, h=h, box=(3.2, 3.2, 3.2), iters=2, seed=5)
    rng = np.random.default_rng(pile)
    cell = np.array([20.0, 20.0, 20.0]) * h + rng.uniform(0.02 * h, 0.98 * h, (pile, 3))
    x = np.concatenate([base.x, cell.astype(np.float32)])
    _check(f"pile {pile}", dataclasses.replace(base, name="pile", x=x, v=np.zeros_like(x)), 2)
