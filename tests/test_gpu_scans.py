"""Cell counts scanned in one launch (up to 8 tiles of 4096 counters), two (up to
4096 tiles) and three, and list builds beside piles on both sides of the size that
gives them their own launch: chained steps against the oracle."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import bit_mismatches, gpu_run, oracle_run

pytestmark = pytest.mark.gpu


def _check(sc, steps, **kw):
    print(f"{sc.n} particles", flush=True)
    got, ref = gpu_run(sc, steps=steps, **kw), oracle_run(sc, steps=steps)
    assert got["num"] == ref["num"]
    assert bit_mismatches(got["x"], ref["x"]) == 0 and bit_mismatches(got["v"], ref["v"]) == 0


# grids of 2^3, 16^3, 32^3, 32*32*64, 64^3 and 512*256*256 cells: 1, 1, 8, 16, 64 and
# 8192 tiles of the search, as many or half of the regrouping
@pytest.mark.parametrize("box", [(0.2, 0.2, 0.2), (1.6, 1.6, 1.6), (3.2, 3.2, 3.2), (3.2, 3.2, 6.4), (6.4, 6.4, 6.4),
                                 (51.2, 25.6, 25.6)])
@pytest.mark.parametrize("unit_width", [1, 16])
def test_scan_forms(box, unit_width):
    if box[0] < 1.0:
        sc = scenes.small_dam(4, 4, 4, h=0.1, box=box, iters=2, seed=8)
    else:
        sc = scenes.small_dam(14, 12, 9, h=0.1, box=box, iters=2, seed=8)
    _check(sc, 3, tile_cap=2048, unit_width=unit_width)


@pytest.mark.parametrize("layers", [38, 40])
def test_list_builds_beside_piles(layers):
    base = scenes.small_dam(64, layers, 32, h=0.1, box=(3.2, 3.2, 3.2), iters=1, seed=9)
    rng = np.random.default_rng(layers)
    near = rng.uniform([0.001, 2.501, 1.101], [0.099, 2.699, 1.299], (900, 3))
    far = rng.uniform([3.2, 2.501, 1.101], [3.2, 2.699, 1.299], (1500, 3))
    x = np.concatenate([base.x, near, far]).astype(np.float32)
    assert (len(x) <= 81920) == (layers == 38)
    _check(dataclasses.replace(base, name="piles", x=x, v=np.zeros_like(x)), 1)
