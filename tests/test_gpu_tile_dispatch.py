"""The edges of the rules that put a step on LDS tiles: the largest state of the
single-workgroup sort and the next one (4,096 and 4,097 particles, that sort
left on), states at and below PBF_TILE_MIN, schedules that replay captured tiled
steps four at a time and one at a time, against the oracle."""
import os

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles

pytestmark = pytest.mark.gpu


def context(p, **env):
    os.environ.update(env)
    try:
        return Particles(p)
    finally:
        for k in env:
            os.environ.pop(k)


@pytest.mark.parametrize("n,tile_min", [(4096, 1), (4097, 1), (4999, 5000), (5000, 5000)])
@pytest.mark.parametrize("schedule", ["flat", "graph"])
def test_dispatch_edges_bit_exact(orc, n, tile_min, schedule):
    k = int(np.ceil(n ** (1 / 3)))
    r = np.random.default_rng(n)
    x = scenes.lattice_block(k, k, k, 0.05, (0.05, 0.05, 0.05))[:n]
    x = (x + r.uniform(-1e-3, 1e-3, x.shape)).astype(np.float32)
    v = r.uniform(-0.3, 0.3, x.shape).astype(np.float32)
    p = scene_params(0.1, 0.05, (0, 0, 0), (1.1, 1.1, 1.1), dt=0.005, max_neighbors=256)
    ref = orc.step(p, x, v, 10, orc.NBR_GRID)
    with context(p, PBF_TILE_MIN=str(tile_min)) as c:
        c.set_schedule(schedule)
        for calls in ((10,), (10,), (4, 1, 5), (1,) * 10):
            c.load(x, v)
            for m in calls:
                c.time_step(nsteps=m)
            for a, b in zip(c.read(), ref):
                assert np.array_equal(a.view(np.uint32), np.asarray(b, np.float32).view(np.uint32))
