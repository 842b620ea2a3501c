"""The graph schedule replays captured steps in every call of one step and of
three or more, one at a time or four: calls of 1 to 50 steps over small,
batched and tiled states, with reads, reloads and changes of dt between, equal
plain launches bit for bit, and so do their lists."""
import os

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles

pytestmark = pytest.mark.gpu


def _context(p, spec=None, **env):
    os.environ.update(env)
    try:
        return Particles(p, scenes=spec)
    finally:
        for k in env:
            os.environ.pop(k)


def _block(n, seed, corner=(0.05, 0.05, 0.05)):
    k = int(np.ceil(n ** (1 / 3)))
    x = scenes.lattice_block(k, k, k, 0.05, corner)[:n]
    r = np.random.default_rng(seed)
    return ((x + r.uniform(-1e-3, 1e-3, x.shape)).astype(np.float32),
            r.uniform(-0.3, 0.3, x.shape).astype(np.float32))


STATES = {
    # name -> (counts per scene, environment of the replaying context)
    "small": ([700], {}),
    "general_sort": ([5000], {}),
    "batch": ([900, 2500, 400], {}),
    "tiles": ([6000], {"PBF_TILE_MIN": "1"}),
}


@pytest.mark.parametrize("name", list(STATES))
def test_calls_of_any_length_equal_plain_launches(name):
    counts, env = STATES[name]
    p = scene_params(0.1, 0.05, (0, 0, 0), (1.2, 1.2, 1.2), dt=0.005, max_neighbors=256)
    spec = None if len(counts) == 1 else [(n, (0, 0, 0), (1.2, 1.2, 1.2)) for n in counts]
    parts = [_block(n, 3 + k) for k, n in enumerate(counts)]
    x, v = (np.concatenate(a) for a in zip(*parts))
    with _context(p, spec, PBF_STEP_GRAPH="0", PBF_TILE_MIN="1000000000") as plain, \
            _context(p, spec, **env) as graph, _context(p, spec, **env) as flat:
        graph.set_schedule("graph")
        for c in (plain, graph, flat):
            c.load(x, v)
        # 3 to 5 steps replay one captured step, 6 and more four at a time from
        # their second call on (2 and 3 replays of four among them), 44 at once.
        for k, n in enumerate((4, 1, 5, 2, 3, 4, 6, 6, 10, 13, 1, 7, 6, 15, 3, 44, 50)):
            dt = p.dt if k < 12 or k > 14 else 0.4 * p.dt
            if k in (7, 13):
                for c in (plain, graph, flat):
                    c.load(x, v)
            for c in (plain, graph, flat):
                c.time_step(dt=dt, nsteps=n)
            ref = plain.read()
            for c in (graph, flat):
                assert all(np.array_equal(a.view(np.uint32), b.view(np.uint32))
                           for a, b in zip(c.read(), ref)), (k, n)
                assert c.neighbor_stats() == plain.neighbor_stats()
        a, b = plain.neighbors(stride=64), graph.neighbors(stride=64)
        assert np.array_equal(a[0], b[0])
        for i, m in enumerate(a[0]):
            assert np.array_equal(a[1][i, :min(m, 64)], b[1][i, :min(m, 64)])
