"""Tiled steps of states with sparse blocks (a lane per particle, in the tiles'
launches), blocks on both sides of the 128 particles from which they take a
tile, sparse and full blocks side by side, and cells that fit no tile at any
level: bit for bit against the oracle, with the lists of the per-lane passes."""
import os

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles

pytestmark = pytest.mark.gpu

H = 0.1
TILES = {"PBF_TILE_MIN": "1", "PBF_NO_SMALL_SORT": "1"}
LANES = {"PBF_TILE_MIN": "1000000000", "PBF_NO_SMALL_SORT": "1", "PBF_WIDE_MAX": "0",
         "PBF_QUAD_MAX": "0", "PBF_DENSE_LIST": "0", "PBF_DENSE_CELL": "0"}


def context(p, env):
    os.environ.update(env)
    try:
        return Particles(p)
    finally:
        for k in env:
            os.environ.pop(k)


def cloud(seed, n, lo, hi):
    return np.random.default_rng(seed).uniform(lo, hi, (n, 3)).astype(np.float32)


def blocks(counts):
    """One block of 5 x 4 x 3 cells per count, with that many particles."""
    c = H * (1.0 + 1.0 / 1024.0)
    return np.concatenate([cloud(20 + k, n, (5 * c * k + 0.01, 0.01, 0.01),
                                 (5 * c * (k + 1) - 0.01, 4 * c - 0.01, 3 * c - 0.01))
                           for k, n in enumerate(counts)])


# name -> (positions, box, max_neighbors)
STATES = {
    "gas": lambda: (cloud(1, 6000, 0.0, 1.9), (1.9, 1.9, 1.9), 128),
    "around_a_tile": lambda: (cloud(2, 4200, 0.0, 1.23), (1.23, 1.23, 1.23), 128),
    "block_counts": lambda: (blocks([1, 63, 127, 128, 129, 512, 513, 0, 64, 300]), (5.1, 0.5, 0.4), 512),
    "spray_over_fluid": lambda: (np.concatenate([
        scenes.lattice_block(26, 12, 22, 0.05, (0.03, 0.03, 0.03)).astype(np.float32),
        cloud(3, 1500, (0.0, 0.65, 0.0), (1.37, 1.83, 1.21))]), (1.37, 1.83, 1.21), 256),
    "fits_no_tile": lambda: (np.concatenate([cloud(4, 2700, 0.52, 0.58), cloud(5, 300, 0.41, 0.73),
                                             cloud(6, 900, 0.0, 1.0)]), (1, 1, 1), 4096),
}


@pytest.mark.parametrize("name", list(STATES))
def test_sparse_states_bit_exact(orc, name):
    x, box, k = STATES[name]()
    p = scene_params(H, H / 2, (0, 0, 0), box, dt=0.002, max_neighbors=k)
    x = np.clip(x, 0, np.asarray(box, np.float32))
    v = np.random.default_rng(11).uniform(-0.3, 0.3, size=x.shape).astype(np.float32)
    ref = orc.step(p, x, v, 2, orc.NBR_GRID)
    lists = []
    for env in (TILES, LANES):
        with context(p, env) as c:
            c.load(x, v)
            c.time_step(nsteps=2)
            for a, b in zip(c.read(), ref):
                assert np.array_equal(a.view(np.uint32), np.asarray(b, np.float32).view(np.uint32))
            counts, ids = c.neighbors(stride=k)
            lists.append(([ids[i, :m].tolist() for i, m in enumerate(counts)], c.neighbor_stats()))
    assert lists[0] == lists[1]
