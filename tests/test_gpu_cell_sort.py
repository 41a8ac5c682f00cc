"""Order inside cells of every size class of the sort (a wave's 64 places, one and
several exchanges beyond it, a full LDS buffer, chunks that are merged): the cell
sort is stable, as the oracle's."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import gpu_run, oracle_run, replace_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(64, 65, 66), (127, 128, 129), (255, 1024, 1025), (2047, 4097), (16384,), (16385,)])
def test_cells_are_sorted_stably(sizes):
    base = scenes.small_dam(6, 5, 4, h=0.1, box=(3.2, 3.2, 3.2), iters=1, seed=2)
    rng = np.random.default_rng(sum(sizes))
    piles = [np.array([1.0 + 0.5 * k, 2.0, 2.0]) + rng.uniform(0.02, 0.08, (n, 3)) for k, n in enumerate(sizes)]
    x = np.concatenate([base.x, *piles]).astype(np.float32)
    rng.shuffle(x)
    sc = replace_params(dataclasses.replace(base, name="cells", x=x, v=np.zeros_like(x)), xsph_on=0, vort_on=0)
    print(f"cells of {sizes}: {sc.n} particles", flush=True)
    got, ref = gpu_run(sc, with_ns=True), oracle_run(sc, want_ns=True)
    assert sorted(np.diff(got["cell_offset"][:-1]))[-len(sizes):] == list(sizes)
    np.testing.assert_array_equal(got["cell_offset"], ref["cell_offset"])
    np.testing.assert_array_equal(got["sorted_index"], ref["sorted_index"])
