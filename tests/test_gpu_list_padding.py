"""The entries past a list's end.  Lists are stored four entries to a word and
walked eight records at a time, so that a last word's unused entries are loaded as
well; those of the final lists name slot 0.  With a particle at NaN there (it hashes
into the first cell) every other particle's sums must still equal the oracle's, by 16,
4 and one lanes a particle."""
from __future__ import annotations

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import bit_mismatches, gpu_run, oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(12, 10, 8), (32, 32, 20), (48, 48, 40)])
def test_record_past_the_end_is_not_used(dims):
    sc = scenes.small_dam(*dims, h=0.1, box=(3.2, 3.2, 3.2), iters=2, seed=5, v_sigma=0.1)
    sc.x[0] = np.nan
    print(f"list padding: {sc.n} particles", flush=True)
    got = gpu_run(sc, with_ns=True)
    ref = oracle_run(sc, want_ns=True)
    assert got["num"] == ref["num"] == sc.n
    np.testing.assert_array_equal(got["sorted_index"], ref["sorted_index"])
    assert got["sorted_index"][0] == 0 and np.isnan(got["x"][0]).all()
    assert np.isfinite(got["v"]).all(axis=1).sum() > sc.n // 2
    assert bit_mismatches(got["x"], ref["x"]) == 0 and bit_mismatches(got["v"], ref["v"]) == 0
