"""States above the size of the LDS tiles that turn from sparse to full and from
full to sparse, by a reload and by moving: whichever passes a step takes, it
gives the bits and the lists of a context without tiles, in calls of one step
(replayed), of several, asynchronous ones and with the graph schedule."""
import os

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles

pytestmark = pytest.mark.gpu

N = 400128


def plain(p):
    os.environ["PBF_TILE_MIN"] = "1000000000"
    try:
        return Particles(p)
    finally:
        os.environ.pop("PBF_TILE_MIN")


def same(a, b):
    return all(np.array_equal(u.view(np.uint32), w.view(np.uint32)) for u, w in zip(a, b))


@pytest.mark.parametrize("schedule", ["flat", "graph"])
def test_states_that_change_their_density(schedule):
    r = np.random.default_rng(9)
    box = 12.0
    p = scene_params(0.1, 0.05, (0, 0, 0), (box,) * 3, dt=0.005, max_neighbors=512)
    p = p.replace(gravity=0.0)
    gas = r.uniform(0, box, (N, 3)).astype(np.float32)
    k = int(np.ceil(N ** (1 / 3)))
    block = scenes.lattice_block(k, k, k, 0.05, (4, 4, 4))[:N].astype(np.float32)
    burst = (40.0 * (block - block.mean(0))).astype(np.float32)   # leaves its blocks sparse
    gather = ((6.0 - gas) * 5.0).astype(np.float32)               # towards the middle
    with plain(p) as a, Particles(p) as b:
        b.set_schedule(schedule)
        for x, v in ((gas, None), (block, None), (gas, None), (block, burst), (gas, gather)):
            for c in (a, b):
                c.load(x, v)
            for n in (1, 1, 1, 40, 1, 1):
                for c in (a, b):
                    c.time_step(nsteps=n)
                assert same(a.read(), b.read()), n
                assert a.neighbor_stats() == b.neighbor_stats()
            for c in (a, b):
                c.step_async(3)
                c.step_async(1)
                c.sync()
            assert same(a.read(), b.read())
            (ca, ia), (cb, ib) = a.neighbors(stride=8), b.neighbors(stride=8)
            assert np.array_equal(ca, cb)
            keep = np.arange(8)[None, :] < np.minimum(ca, 8)[:, None]
            assert np.array_equal(ia[keep], ib[keep])


def test_which_passes_run():
    """Sparse states stay off the tiles and full ones take them, from the first
    step after a load on; a state that spreads leaves them."""
    r = np.random.default_rng(2)
    p = scene_params(0.1, 0.05, (0, 0, 0), (12.0,) * 3, dt=0.005, max_neighbors=512)
    p = p.replace(gravity=0.0)
    gas = r.uniform(0, 12, (N, 3)).astype(np.float32)
    k = int(np.ceil(N ** (1 / 3)))
    block = scenes.lattice_block(k, k, k, 0.05, (4, 4, 4))[:N].astype(np.float32)
    burst = (40.0 * (block - block.mean(0))).astype(np.float32)
    with Particles(p) as c, plain(p) as off:
        assert not c.tiled()
        for x, v, first, last in ((gas, None, False, False), (block, None, True, True),
                                  (gas, None, False, False), (block, burst, True, False)):
            c.load(x, v)
            assert not c.tiled()
            c.time_step()
            assert c.tiled() == first
            c.time_step(nsteps=20)
            c.time_step()
            assert c.tiled() == last
        off.load(block, None)
        off.time_step()
        assert not off.tiled()
