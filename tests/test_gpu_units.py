"""Work items of the search and of the final passes, listed tile by tile while
the cell counts are scanned: at every run width from one cell to the widest, on
a scene with empty runs, ragged ends and a run of several 256-particle chunks,
their number must be what the splitting rule gives on the cell offsets, and the
step must equal the oracle bit for bit (every particle in exactly one item)."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import bit_mismatches, gpu_run, oracle_run

pytestmark = pytest.mark.gpu

CHUNK = 256


def dense_run_scene():
    """A ragged lattice and a clump of 700 particles inside two cells."""
    base = scenes.small_dam(13, 9, 7, h=0.1, box=(3.2, 1.6, 1.6), iters=2, seed=4)
    rng = np.random.default_rng(9)
    clump = np.array([2.05, 0.95, 0.95]) + rng.uniform(0.0, 0.1, (700, 3)) * np.array([1.0, 0.4, 0.4])
    x = np.concatenate([base.x, clump.astype(np.float32)]).astype(np.float32)
    return dataclasses.replace(base, name="dense_run", x=x, v=np.zeros_like(x))


def expected_items(off, uw, budget):
    n = 0
    for k in range(0, off.size - 2, uw):
        seg = int(off[k + uw]) - int(off[k])
        if seg == 0:
            continue
        w = uw
        while w > 1 and 9 * (w + 2) * seg > budget * uw:
            w >>= 1
        for q in range(k, k + uw, w):
            n += -(-(int(off[q + w]) - int(off[q])) // CHUNK)
    return n


@pytest.mark.parametrize("unit_width", [1, 2, 8, 32])
@pytest.mark.parametrize("tile_cap", [256, 4096])
def test_search_items_cover_every_particle(unit_width, tile_cap):
    sc = dense_run_scene()
    got = gpu_run(sc, tile_cap=tile_cap, unit_width=unit_width, with_ns=True)
    ref = oracle_run(sc, want_ns=True)
    off = got["cell_offset"].astype(np.int64)
    assert got["stats"]["units"] == expected_items(off, unit_width, tile_cap * 3 // 4)
    np.testing.assert_array_equal(got["neighbor_count"], ref["neighbor_count"][: got["num"]])
    assert got["num"] == ref["num"]
    assert bit_mismatches(got["x"], ref["x"]) == 0 and bit_mismatches(got["v"], ref["v"]) == 0
