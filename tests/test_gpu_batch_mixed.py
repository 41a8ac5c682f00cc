"""Scenes of one batch with different tensile corrections (exponents 4, 3 and 1,
and the reference's form), box sizes and passes, several of them within one wave:
each scene's step must equal the oracle's plain step of that scene."""
from __future__ import annotations

import pytest

from ssf_pbf_cuda_amd import scenes

from helpers import replace_params
from test_gpu_batch import _check_against_oracle, _run_batch

pytestmark = pytest.mark.gpu

KINDS = [
    dict(),
    dict(scorr_n=3, scorr_k=0.02),
    dict(scorr_n=1, xsph_on=0),
    dict(scorr_mode=scenes.SCORR_REFERENCE, relaxation=6000.0),
    dict(vort_on=0),
    dict(scorr_n=4, scorr_k=0.05, xsph_parameter=0.05),
]


# 18 scenes of 24 particles, 432 in all, and 6 of 3,025 (16 and 4 lanes a particle);
# 6 of 15,000 (one lane)
@pytest.mark.parametrize("dims,copies", [((3, 2, 4), 3), ((11, 11, 25), 1), ((25, 25, 24), 1)])
def test_mixed_scenes_bit_exact(dims, copies):
    nx, ny, nz = dims
    scs = []
    for c in range(copies):
        for i, kw in enumerate(KINDS):
            box = (1.6, 1.6, 1.6) if max(dims) <= 11 else (3.2, 3.2, 3.2)
            sc = scenes.small_dam(nx, ny, nz, h=0.1, box=box, iters=3, seed=7 * c + i, v_sigma=0.2)
            scs.append(replace_params(sc, **kw))
    print(f"mixed batch: {len(scs)} scenes, {sum(s.n for s in scs)} particles", flush=True)
    _check_against_oracle(scs, _run_batch(scs, 2), 2)
