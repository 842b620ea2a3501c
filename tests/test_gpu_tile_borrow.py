"""A context whose loaded state steps on LDS tiles, with pbf_step_device_noalloc
calls on other states in between: the loaded state's particles, lists and cells
stay as they were, and the borrowed run gives the bits of the allocating path."""
import os

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles
from test_zz_no_alloc import noalloc_path, same_bits

pytestmark = pytest.mark.gpu


def context(p, tile_min):
    os.environ["PBF_TILE_MIN"] = str(tile_min)
    os.environ["PBF_NO_SMALL_SORT"] = "1"
    try:
        return Particles(p)
    finally:
        os.environ.pop("PBF_TILE_MIN")
        os.environ.pop("PBF_NO_SMALL_SORT")


def block(side, seed):
    x = scenes.lattice_block(side, side, side, 0.05, (0.05, 0.05, 0.05))
    return (x + np.random.default_rng(seed).uniform(-1e-3, 1e-3, x.shape)).astype(np.float32)


def lists(c, stride):
    counts, ids = c.neighbors(stride=stride)
    return [ids[i, :k].tolist() for i, k in enumerate(counts)], c.cells().tolist(), c.neighbor_stats()


def check_state_kept(tile_min, n_borrowed):
    p = scene_params(0.1, 0.05, (0, 0, 0), (1, 1, 1), dt=0.005, max_neighbors=128)
    x, y = block(15, 1), block(18, 2)[:n_borrowed]
    v = np.random.default_rng(3).uniform(-0.5, 0.5, y.shape).astype(np.float32)
    with Particles(p) as c:
        c.load(y, v)
        c.time_step(dt=p.dt, nsteps=3)
        ref = c.read()[:2]
    with context(p, tile_min) as c:
        c.load(x, None)
        c.time_step(nsteps=2)
        before, state = lists(c, 128), c.read()
        got = noalloc_path(c, y, v, 3, p.dt)
        assert all(same_bits(a, b) for a, b in zip(got, ref))
        assert lists(c, 128) == before
        assert all(same_bits(a, b) for a, b in zip(c.read(), state))


@pytest.mark.parametrize("n", [500, 1999])
def test_lists_survive_a_borrowed_run_below_the_tile_threshold(n):
    check_state_kept(2000, n)


@pytest.mark.parametrize("n", [1, 1000, 3375, 5832])
def test_borrowed_runs_take_no_tiles_of_the_loaded_state(n):
    """The workspace holds no tiles and no queues, so its run keeps the other
    passes, also for more particles than the context's tiles are sized for."""
    check_state_kept(1, n)
