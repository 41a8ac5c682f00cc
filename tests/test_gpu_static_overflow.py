"""The allocation-free step with more blocks of overflowing final lists than its 64
overflow slots: the sums of the blocks left over go cell by cell in the passes, by 16
lanes a particle (up to 16,384 particles) or four, with and without cells of more
than 64 particles.  The state must equal the oracle's."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import bit_mismatches, gpu_run, oracle_run
from test_zz_no_alloc import _static_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_cell,cells", [(31, (8, 8, 6)), (31, (10, 10, 10)), (440, (3, 3, 3)), (1111, (3, 3, 3))])
def test_more_overflowing_blocks_than_slots(per_cell, cells):
    h = 0.1
    base = scenes.small_dam(4, 4, 4, h=h, box=(1.6, 1.6, 1.6), iters=1, scorr_k=0.001)
    rng = np.random.default_rng(per_cell)
    at = np.stack(np.meshgrid(*[np.arange(3, 3 + c) for c in cells], indexing="ij"), -1).reshape(-1, 3)
    x = (np.repeat(at, per_cell, axis=0) + rng.uniform(0.02, 0.98, (len(at) * per_cell, 3))) * h
    rng.shuffle(x)
    v = rng.normal(0.0, 0.05, x.shape)
    sc = dataclasses.replace(base, name="dense", x=x.astype(np.float32), v=v.astype(np.float32))
    over = gpu_run(sc)["stats"]["list_overflow"]
    print(f"static step: {sc.n} particles, {over} overflowing", flush=True)
    assert over > 64 * 64
    sx, sv = _static_step(sc)
    ref = oracle_run(sc)
    assert ref["num"] == sc.n
    assert bit_mismatches(sx, ref["x"]) == 0 and bit_mismatches(sv, ref["v"]) == 0
