"""The per-cell sums of blocks with overflowing final lists, by rows of 16 lanes or
by threads, on both sides of the lines between the two (overflowing particles above 64
times the largest cell, which counts as 64 at least, above 24 times where their blocks of
64 are full, or above 655,360): without cells of more than 64 particles, with one, with
full ones, and in a batch.  Each state must equal the oracle's plain step."""
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


# box, particles of one point, by threads
CASES = {
    "few": (30, (0.4, 0.4, 0.4), 0, False),
    "small_cells": (30, (0.8, 0.8, 0.8), 0, True),
    "one_larger_cell": (30, (0.8, 0.8, 0.8), 700, False),
    "full_cells": (700, (0.4, 0.4, 0.4), 0, True),
    "few_full_cells": (700, (0.4, 0.2, 0.2), 0, False),
    "many_blocks": (15, (6.4, 3.2, 3.2), 7000, False),
    "below_the_line": (17, (3.2, 3.2, 3.2), 10500, False),
    "above_the_line": (30, (3.2, 3.2, 3.2), 16000, True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_both_forms(name):
    per_cell, box, point, threads = CASES[name]
    sc = filled(per_cell, box)
    sc.x[:point] = sc.x[0]
    got = gpu_run(sc, with_ns=True)
    over, most = got["stats"]["list_overflow"], np.diff(got["cell_offset"][:-1].astype(np.int64)).max()
    print(f"{name}: {sc.n} particles, {over} overflowing, cells of up to {most}", flush=True)
    assert over > 0 and (most > 64) == (point > 0 or per_cell > 64)
    if name == "full_cells":
        assert over == sc.n and 24 * most < over <= 64 * most
    else:
        assert (over > min(LINE, 64 * max(64, most))) == threads
        assert threads or over < max(24 * max(64, most), 56 * (sc.n // 64))
    if name == "many_blocks":
        assert sc.n > LINE
    ref = oracle_run(sc)
    assert got["num"] == ref["num"]
    assert bit_mismatches(got["x"], ref["x"]) == 0 and bit_mismatches(got["v"], ref["v"]) == 0


@pytest.mark.parametrize("point", [0, 300])
def test_threads_in_a_batch(point):
    scs = [filled(30, (3.2, 3.2, 1.6), seed=s) for s in (5, 6)]
    scs.append(scenes.small_dam(12, 10, 8, iters=1))
    if point:
        scs[0].x[:point] = scs[0].x[0]  # coincident: a cell of more than 64 particles
    print(f"batch of {[s.n for s in scs]} particles", flush=True)
    _check_against_oracle(scs, _run_batch(scs, 1), 1)
