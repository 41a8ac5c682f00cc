"""The autotuner chooses by time, and tile_cap moves statistics only: it stays as it
was set, and the statistics of the next step follow it and the returned width."""
from __future__ import annotations

import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import gpu_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile_cap", [0, 512, 2048])
def test_autotune_keeps_tile_cap(tile_cap):
    import torch

    from ssf_pbf_cuda_amd import pbfx

    sc = scenes.small_dam(32, 32, 32, box=(3.2, 3.2, 1.6), iters=2)
    solver = pbfx.Solver.for_scene(sc)
    solver.set_tuning(tile_cap, 16)
    x, v = torch.from_numpy(sc.x).cuda(), torch.from_numpy(sc.v).cuda()
    xs, vs = torch.empty_like(x), torch.empty_like(v)
    tile, width = solver.autotune(x, v, sc.n, sc.area_lo, sc.area_hi, sc.iters, xs, vs)
    assert tile == tile_cap and width in (4, 8, 16, 32)
    solver.step(x, v, sc.n, sc.area_lo, sc.area_hi, sc.iters)
    got = solver.stats()
    solver.close()
    ref = gpu_run(sc, tile_cap=tile_cap, unit_width=width)["stats"]
    for k in ("units", "slow_units", "slow_particles", "max_tile", "final_units"):
        assert got[k] == ref[k], (k, got[k], ref[k])
