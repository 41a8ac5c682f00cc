"""Lists built by groups of eight lanes, and list sums by several lanes per
particle, at the sizes where their steps end: cells of 0, 1, 7, 8, 9, 15, 16,
17, 33, 64 and 65 particles (one step, two, more, a big cell), lists of 1, 29
and 63 entries and exactly full ones, grids one and two cells wide (the 27
cells repeat), and particle counts around the lane rules (16 lanes up to
16,384 particles, four up to 81,920, one above).  Lists, positions and
velocities must equal the oracle bit for bit."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import bit_mismatches, gpu_run, oracle_run, replace_params

pytestmark = pytest.mark.gpu

COUNTS = [0, 1, 7, 8, 9, 15, 16, 17, 33, 64, 65, 8, 8, 3]


def cells_scene(box, seed=2, **params):
    """Cells of the box filled with COUNTS in turn (spread over each cell)."""
    h = 0.1
    base = scenes.small_dam(4, 4, 4, h=h, box=box, iters=2, seed=seed, **params)
    rng = np.random.default_rng(seed)
    dims = [max(1, int(round(b / h))) for b in box]
    pts, k = [], 0
    for z in range(dims[2]):
        for y in range(dims[1]):
            for x in range(dims[0]):
                n = COUNTS[k % len(COUNTS)]
                k += 1
                pts.append((np.array([x, y, z]) + rng.uniform(0.02, 0.98, (n, 3))) * h)
    x = np.concatenate(pts)
    rng.shuffle(x)
    x = x.astype(np.float32)
    v = rng.normal(0.0, 0.05, x.shape).astype(np.float32)
    return dataclasses.replace(base, name="cells", x=x, v=v)


def check(sc, **kw):
    got = gpu_run(sc, with_ns=True, **kw)
    ref = oracle_run(sc, want_ns=True)
    nl, m = got["num"], sc.params.max_pair
    assert nl == ref["num"]
    np.testing.assert_array_equal(got["neighbor_count"], ref["neighbor_count"][:nl])
    np.testing.assert_array_equal(got["neighbors"], ref["neighbors"].reshape(-1, m)[:nl])
    assert bit_mismatches(got["x"], ref["x"]) == 0 and bit_mismatches(got["v"], ref["v"]) == 0
    return got


@pytest.mark.parametrize("max_pair", [2, 30, 64])
@pytest.mark.parametrize("counts", ["mixed", "no_big_cell"])
def test_cells_of_every_step_count(max_pair, counts):
    sc = cells_scene((0.7, 0.6, 0.5), scorr_k=0.001)
    if counts == "no_big_cell":  # the kernels of a step without cells of more than 64 particles
        sc = dataclasses.replace(sc, x=sc.x[::3].copy(), v=sc.v[::3].copy())
    check(replace_params(sc, max_pair=max_pair))


@pytest.mark.parametrize("box", [(0.1, 0.1, 0.1), (0.25, 0.15, 0.1), (0.35, 0.1, 0.3)])
def test_grids_of_one_and_two_cells(box):
    check(cells_scene(box, seed=3, scorr_k=0.001))


@pytest.mark.parametrize("n", [16384, 16385, 81920, 81921])
def test_lane_rules(n):
    sc = scenes.small_dam(48, 48, 36, h=0.1, box=(3.2, 3.2, 1.6), iters=2, seed=5, scorr_k=0.001, v_sigma=0.1)
    keep = np.sort(np.random.default_rng(n).permutation(sc.n)[:n])
    check(dataclasses.replace(sc, x=sc.x[keep].copy(), v=sc.v[keep].copy()))


@pytest.mark.parametrize("per_cell", [17, 33, 64, 65])
def test_overflowing_final_lists(per_cell):
    """More than 64 pairs a particle: the sums go cell by cell, 16 candidates a
    step, with and without cells of more than 64 particles."""
    h = 0.1
    base = scenes.small_dam(4, 4, 4, h=h, box=(0.5, 0.4, 0.4), iters=1, seed=3, scorr_k=0.001)
    rng = np.random.default_rng(per_cell)
    x = np.concatenate([(np.array([i % 5, i // 5 % 4, i // 20]) + rng.uniform(0.05, 0.95, (per_cell, 3))) * h
                        for i in range(80)]).astype(np.float32)
    got = check(dataclasses.replace(base, x=x, v=rng.normal(0.0, 0.05, x.shape).astype(np.float32)))
    print(per_cell, got["stats"]["list_overflow"], flush=True)
    assert got["stats"]["list_overflow"] > 0
