"""Collision sweeps that never settle (particles resting on walls in the wild
flow, spheres against planes): the solver jumps to the end of a repeating
cycle, and must leave what the oracle's sweep-by-sweep loop leaves, at odd and
even caps."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import bit_mismatches, gpu_run, oracle_run, replace_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_sweeps", [1, 2, 3, 4, 7, 32, 33])
@pytest.mark.parametrize("spheres", [False, True])
def test_capped_sweeps_match_the_oracle(max_sweeps, spheres):
    sc = replace_params(scenes.small_dam(14, 12, 9, h=0.1, box=(1.6, 0.8, 0.8), iters=4, seed=6), max_sweeps=max_sweeps)
    if spheres:
        sc = dataclasses.replace(sc, inner_spheres=np.array([[0.8, 0.4, 0.4, 0.95]], np.float32),
                                 outer_spheres=np.array([[1.2, 0.1, 0.4, 0.2]], np.float32))
    got, ref = gpu_run(sc, steps=3), oracle_run(sc, steps=3)
    print(max_sweeps, spheres, got["stats"]["sweep_cap_hits"], flush=True)
    assert got["num"] == ref["num"]
    assert bit_mismatches(got["x"], ref["x"]) == 0 and bit_mismatches(got["v"], ref["v"]) == 0
    assert got["stats"]["max_sweeps_used"] <= max_sweeps
