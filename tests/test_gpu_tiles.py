"""List passes over LDS tiles, forced on small states (PBF_TILE_MIN=1), bit for
bit against the oracle: grids that the blocks of 5 x 4 x 3 cells do not divide,
counts around a wave and around the largest state of the single-workgroup
sort, blocks cut into parts and cells that stand out of their tile (the
queue), sparse blocks (the queue), coincident pairs and pairs closer than
EPS_D (the general terms), the graph schedule and one-step calls; the exported
lists equal those of the per-lane passes, and an overflow is reported."""
import os

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles, PbfError

pytestmark = pytest.mark.gpu

TILES = {"PBF_TILE_MIN": "1", "PBF_NO_SMALL_SORT": "1"}
LANES = {"PBF_TILE_MIN": "1000000000", "PBF_NO_SMALL_SORT": "1", "PBF_WIDE_MAX": "0",
         "PBF_QUAD_MAX": "0", "PBF_DENSE_LIST": "0", "PBF_DENSE_CELL": "0"}


def bits_equal(a, b):
    a = np.ascontiguousarray(a, np.float32)
    b = np.ascontiguousarray(b, np.float32)
    return a.shape == b.shape and np.array_equal(a.view(np.uint32), b.view(np.uint32))


def context(p, env=TILES):
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        return Particles(p)
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v


def params(box, h=0.1, **kw):
    return scene_params(h, h / 2, (0, 0, 0), box, dt=0.005, **kw)


def cloud(seed, n, lo, hi):
    return np.random.default_rng(seed).uniform(lo, hi, size=(n, 3)).astype(np.float32)


def lattice(nx, ny, nz, spacing, corner, seed):
    x = scenes.lattice_block(nx, ny, nz, spacing, corner)
    return (x + np.random.default_rng(seed).uniform(-1e-3, 1e-3, x.shape)).astype(np.float32)


def close_pairs():
    """A lattice whose first particles sit on others: 8 coincident pairs, and
    near the origin (where floats resolve it) pairs 1e-12 and 3e-11 apart."""
    x = lattice(14, 14, 14, 0.05, (0.1, 0.1, 0.1), 5)
    x[:8] = x[8:16]
    x[20] = (0.0, 0.3, 0.3)
    x[21] = (1e-12, 0.3, 0.3)
    x[22] = (0.0, 0.5, 0.3)
    x[23] = (3e-11, 0.5, 0.3)
    return x


# name -> (positions, box, max_neighbors)
STATES = {
    "one": lambda: (np.array([[0.3, 0.4, 0.5]], np.float32), (1, 1, 1), 64),
    "sparse": lambda: (cloud(1, 900, 0.02, 2.9), (3, 3, 3), 64),
    "wave_edge": lambda: (lattice(5, 5, 13, 0.05, (0.02, 0.02, 0.02), 2), (0.7, 0.7, 0.9), 128),
    "odd_grid": lambda: (lattice(23, 17, 11, 0.05, (0.01, 0.01, 0.01), 3), (1.3, 1.05, 0.62), 128),
    "above_small_sort": lambda: (lattice(13, 14, 15, 0.05, (0.1, 0.1, 0.1), 4)[:2561], (1, 1, 1), 128),
    # Three times rest density throughout: blocks cut into parts.
    "dense": lambda: (lattice(27, 27, 27, 0.035, (0.02, 0.02, 0.02), 6), (1, 1, 1), 512),
    # 600 particles in one cell of a lattice, and a clump across a block's edge.
    "spike": lambda: (np.concatenate([lattice(16, 16, 16, 0.05, (0.05, 0.05, 0.05), 7),
                                      cloud(8, 600, 0.41, 0.48), cloud(9, 300, 0.47, 0.56)]),
                      (1, 1, 1), 2048),
    "close_pairs": lambda: (close_pairs(), (1, 1, 1), 128),
}


@pytest.mark.parametrize("name", list(STATES))
def test_tiled_steps_bit_exact(orc, name):
    x, box, k = STATES[name]()
    p = params(box, max_neighbors=k)
    v = np.random.default_rng(11).uniform(-0.3, 0.3, size=x.shape).astype(np.float32)
    if name == "close_pairs":
        # The pairs stay as close as they were loaded.
        p = p.replace(gravity=0.0)
        v[:] = 0.0
    ox, ov, orho = orc.step(p, x, v, 3, orc.NBR_GRID)
    with context(p) as c:
        c.load(x, v)
        c.time_step(nsteps=3)
        gx, gv, grho = c.read()
        assert bits_equal(gx, ox) and bits_equal(gv, ov) and bits_equal(grho, orho)
        # One-step calls (the second and third replay a captured step) and
        # the graph schedule.
        c.load(x, v)
        for _ in range(3):
            c.time_step()
        assert all(bits_equal(a, b) for a, b in zip(c.read(), (ox, ov, orho)))
        c.set_schedule("graph")
        c.load(x, v)
        c.time_step(nsteps=3)
        assert all(bits_equal(a, b) for a, b in zip(c.read(), (ox, ov, orho)))


@pytest.mark.parametrize("name", ["sparse", "odd_grid", "dense", "spike"])
def test_exported_lists_equal_the_per_lane_ones(name):
    x, box, k = STATES[name]()
    p = params(box, max_neighbors=k)
    got = []
    for env in (TILES, LANES):
        with context(p, env) as c:
            c.load(x, None)
            c.time_step()
            counts, ids = c.neighbors(stride=k)
            got.append((counts, [ids[i, :counts[i]].tolist() for i in range(len(x))],
                        c.neighbor_stats()))
    assert np.array_equal(got[0][0], got[1][0])
    assert got[0][1] == got[1][1]
    assert got[0][2] == got[1][2]


def test_overflow_is_reported():
    x, box, _ = STATES["dense"]()
    with context(params(box, max_neighbors=40)) as c:
        c.load(x, None)
        with pytest.raises(PbfError) as e:
            c.time_step()
        assert e.value.code == -3
