"""A scene so large and dense that nearly every block of 64 particles overflows its
final lists (more than 20,480 blocks): the per-cell sums by a thread per cell,
against the oracle."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import bit_mismatches, gpu_run, oracle_run, replace_params

pytestmark = pytest.mark.gpu


def dense_scene(n=1_400_000, seed=3):
    rng = np.random.default_rng(seed)
    base = scenes.small_dam(4, 4, 4, h=0.1, box=(6.4, 3.2, 3.2), iters=1)
    x = rng.uniform([0.0, 0.0, 0.0], [6.4, 3.2, 3.2], (n, 3)).astype(np.float32)
    x[:300] = x[0]  # coincident
    sc = dataclasses.replace(base, name="dense", x=x, v=np.zeros_like(x))
    return replace_params(sc, relaxation=1.0e9, scorr_k=1.0e-6)  # the particles hardly move


def test_many_overflows_bit_exact():
    sc = dense_scene()
    print(f"{sc.n} particles", flush=True)
    got = gpu_run(sc)
    print(got["stats"], flush=True)
    assert got["stats"]["list_overflow"] > 20480 * 64
    ref = oracle_run(sc)
    assert got["num"] == ref["num"]
    assert bit_mismatches(got["x"], ref["x"]) == 0 and bit_mismatches(got["v"], ref["v"]) == 0
