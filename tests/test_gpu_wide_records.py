"""A context of 2^28 slots, from which on a record's byte offset passes 32 bits and
the list builds and list walks load records by plain addresses: piles in one launch,
16 and four lanes a particle, one lane a particle, and piles in launches of their own.
Lists and state must equal the oracle's.  The context takes 264 GB."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import bit_mismatches, gpu_run, oracle_run
from test_gpu_aliased_piles import aliased_scene

pytestmark = pytest.mark.gpu

WIDE = 1 << 28


def piles_in_a_dam():
    """aliased_scene's piles with a dam of 90,000 particles above them."""
    sc = aliased_scene(seed=15)
    dam = scenes.small_dam(60, 30, 50, box=(3.2, 3.2, 3.2), iters=2, seed=6)
    x = np.concatenate([sc.x, (dam.x + np.float32([0.05, 1.6, 0.05])).astype(np.float32)])
    return dataclasses.replace(sc, x=x, v=np.zeros_like(x))


SCENES = {
    "piles": lambda: aliased_scene(seed=15),
    "four_lanes": lambda: scenes.small_dam(32, 32, 20, box=(3.2, 3.2, 3.2), iters=2, seed=5, v_sigma=0.1),
    "one_lane": lambda: scenes.small_dam(48, 48, 40, box=(3.2, 3.2, 3.2), iters=2, seed=5, v_sigma=0.1),
    "piles_one_lane": piles_in_a_dam,
}


@pytest.mark.parametrize("name", list(SCENES))
def test_records_past_32_bit_offsets(name):
    import torch

    if torch.cuda.mem_get_info()[0] < 275e9:
        pytest.skip("needs 275 GB of free GPU memory")
    sc = SCENES[name]()
    print(f"wide records: {name}, {sc.n} particles", flush=True)
    got = gpu_run(sc, with_ns=True, capacity=WIDE)
    torch.cuda.empty_cache()
    ref = oracle_run(sc, want_ns=True)
    nl, m = got["num"], sc.params.max_pair
    assert nl == ref["num"]
    if "piles" in name:
        assert got["stats"]["heavy_builds"] > 0 and got["stats"]["list_overflow"] > 0
    np.testing.assert_array_equal(got["neighbor_count"], ref["neighbor_count"][:nl])
    np.testing.assert_array_equal(got["neighbors"], ref["neighbors"].reshape(-1, m)[:nl])
    assert bit_mismatches(got["x"], ref["x"]) == 0 and bit_mismatches(got["v"], ref["v"]) == 0
