"""Density over the last step's lists at positions that leave the fast root
(coincident, closer than 2^-48, not finite) and at list lengths around the eight
entries loaded together: bit for bit the oracle's."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import pyoracle as orc
from ssf_pbf_cuda_amd import scenes
from tests.helpers import replace_params
from tests.test_gpu_diagnostics import _solver_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_pair", [2, 7, 8, 9, 64])
@pytest.mark.parametrize("odd", [False, True])
def test_density_lists_and_ranges(max_pair, odd):
    import torch

    sc = replace_params(scenes.small_dam(11, 9, 7), max_pair=max_pair)
    print(f"density: n={sc.n} max_pair={max_pair} odd={odd}", flush=True)
    solver, x, v, _, _, num = _solver_run(sc, 1)
    r = orc.step(sc, want_ns=True)
    xs = r["x"].copy()
    if odd:
        nb = r["neighbors"].reshape(-1, max_pair)
        rng = np.random.default_rng(max_pair)
        at = rng.choice(num, 24, replace=False)
        for k, i in enumerate(at):
            j = nb[i][nb[i] != 0xFFFFFFFF]
            j = int(j[k % len(j)]) if len(j) else int(i)
            if k % 4 == 0:
                xs[j] = xs[i]
            elif k % 4 == 1:
                xs[i] = 0.0
                xs[j] = np.float32(2.0) ** np.float32(-49 - k)
            elif k % 4 == 2:
                xs[i, k % 3] = np.nan
            else:
                xs[i, k % 3] = np.inf
    rho = torch.zeros(num, dtype=torch.float32, device="cuda")
    solver.density(torch.from_numpy(xs).cuda(), rho)
    torch.cuda.synchronize()
    ref = orc.density(sc, xs, r["neighbors"])
    got = rho.cpu().numpy()
    assert np.array_equal(got.view(np.uint32)[~np.isnan(ref)], ref.view(np.uint32)[~np.isnan(ref)])
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    solver.close()
