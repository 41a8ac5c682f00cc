"""A batch of more than 81,920 particles whose lists of steps with big cells have
launches of their own: two scenes of piles that the wrapping hash puts into one cell,
beside and between plain dams, with lists long enough for a whole wave each.  Every
scene must equal the oracle's plain step of it."""
from __future__ import annotations

import numpy as np
import pytest

from ssf_pbf_cuda_amd import scenes

from test_gpu_aliased_piles import aliased_scene
from test_gpu_batch import _check_against_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1, 2])
def test_piles_in_a_large_batch(steps):
    import torch

    from ssf_pbf_cuda_amd import pbfx

    scs = [scenes.small_dam(40, 32, 32, box=(6.4, 3.2, 3.2), seed=3, iters=2, v_sigma=0.1),
           aliased_scene(seed=15),
           scenes.small_dam(5, 3, 3, seed=4, iters=2),
           aliased_scene(far=1500, near=900, point=300, seed=14),
           scenes.small_dam(40, 32, 32, box=(6.4, 3.2, 3.2), seed=5, iters=2)]
    counts = [s.n for s in scs]
    assert sum(counts) > 81920
    print(f"batch with piles: {counts}", flush=True)
    solver = pbfx.BatchSolver(scs)
    x = torch.from_numpy(np.concatenate([s.x for s in scs])).cuda()
    v = torch.from_numpy(np.concatenate([s.v for s in scs])).cuda()
    for k in range(steps):
        counts = solver.batch_step(x, v, counts, scs[0].iters)
        st = solver.stats()
        print({k: st[k] for k in ("heavy_builds", "heavy_search", "list_overflow")}, flush=True)
        assert st["list_overflow"] > 0
        if k == 0:  # the piles burst in this step
            assert st["heavy_builds"] > 0 and st["heavy_search"] > 0
    end = np.cumsum(counts)
    xs, vs = x.cpu().numpy(), v.cpu().numpy()
    solver.close()
    res = [(xs[e - n:e], vs[e - n:e], n) for e, n in zip(end, counts)]
    _check_against_oracle(scs, res, steps)
