"""Ray batches at the sizes where the traversal kernels split their work
differently, against the oracle: hits bit for bit (the kernels only hand rays
out differently; each ray's own arithmetic does not change)."""
import os

import numpy as np
import pytest

from bulbit_amd import scenes

THREADS = max(1, min(16, len(os.sched_getaffinity(0))))


@pytest.fixture(scope="module")
def small():
    from bulbit_amd.gpu import GpuScene
    from oracle import OracleScene

    sc, _ = scenes.icosphere_scene(level=3)
    return GpuScene(sc), OracleScene(sc)


# one ray; below, at and past the fewest rays a wave starts with (8); one
# wave and one block more; past 8 per wave of a full grid (some 6,000 to 8,000
# waves); and past 128 per wave, where the shared counter takes over
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 7, 8, 9, 64, 65, 129, 70001, 1_050_001])
@pytest.mark.parametrize("any_hit", [False, True])
def test_batch_sizes(small, n, any_hit):
    g, o = small
    bmin, bmax = o.world_bounds()
    rays = scenes.random_rays(bmin, bmax, n, seed=n, t_max=3.0 if any_hit else np.inf)
    hits, _ = g.trace(rays, any_hit=any_hit)
    want, _ = o.trace(rays, any_hit=any_hit, threads=THREADS)
    assert np.array_equal(hits["prim"], want["prim"])
    if not any_hit:
        for f in ("t", "u", "v"):
            assert np.array_equal(hits[f].view(np.int32), want[f].view(np.int32)), f
