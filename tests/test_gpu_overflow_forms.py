"""The per-cell sums of blocks with overflowing final lists, on both sides of the
655,360 overflowing particles at which k_ovf_part goes from rows of 16 lanes to a
thread per cell: fewer particles than that in all, fewer overflowing ones in more than
10,240 blocks, and more, without cells of more than 64 particles; and, in a batch, more
with and without such cells.  Each state must equal the oracle's plain step."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import bit_mismatches, gpu_run, oracle_run, replace_params
from test_gpu_batch import _check_against_oracle, _run_batch

pytestmark = pytest.mark.gpu

LINE = 655360


def filled(per_cell, box, seed=3):
    """per_cell particles in every cell of the box, which hardly move."""
    h = 0.1
    base = scenes.small_dam(4, 4, 4, h=h, box=box, iters=1)
    dims = [int(round(b / h)) for b in box]
    cell = np.stack(np.meshgrid(*[np.arange(d) for d in dims], indexing="ij"), -1).reshape(-1, 3)
    rng = np.random.default_rng(seed)
    x = (np.repeat(cell, per_cell, axis=0) + rng.uniform(0.02, 0.98, (len(cell) * per_cell, 3))) * h
    rng.shuffle(x)
    x = x.astype(np.float32)
    sc = dataclasses.replace(base, name="filled", x=x, v=np.zeros_like(x))
    return replace_params(sc, relaxation=1.0e9, scorr_k=1.0e-6)


@pytest.mark.parametrize("per_cell,width", [(19, 3.2), (15, 6.4), (30, 3.2)])
def test_both_forms_without_big_cells(per_cell, width):
    sc = filled(per_cell, (width, 3.2, 3.2))
    got = gpu_run(sc, with_ns=True)
    over = got["stats"]["list_overflow"]
    print(f"{sc.n} particles, {over} overflowing", flush=True)
    assert np.diff(got["cell_offset"][:-1].astype(np.int64)).max() <= 64
    if per_cell == 19:
        assert 0 < over <= sc.n < LINE
    elif per_cell == 15:
        assert sc.n > LINE * 1.4 and LINE // 4 < over < LINE
    else:
        assert over > LINE
    ref = oracle_run(sc)
    assert got["num"] == ref["num"]
    assert bit_mismatches(got["x"], ref["x"]) == 0 and bit_mismatches(got["v"], ref["v"]) == 0


@pytest.mark.parametrize("point", [0, 300])
def test_threads_per_cell_in_a_batch(point):
    scs = [filled(30, (3.2, 3.2, 1.6), seed=s) for s in (5, 6)]
    scs.append(scenes.small_dam(12, 10, 8, iters=1))
    if point:
        scs[0].x[:point] = scs[0].x[0]  # coincident: a cell of more than 64 particles
    print(f"batch of {[s.n for s in scs]} particles", flush=True)
    _check_against_oracle(scs, _run_batch(scs, 1), 1)
