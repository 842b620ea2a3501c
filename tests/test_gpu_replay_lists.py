"""Lists, cells and neighbour counts after one-step calls that replay a captured
step: after a reload, after another state and after a snapshot, with both
schedules that replay, on tiles and without, they are those of plain launches
(PBF_STEP_GRAPH=0)."""
import os

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles, PbfError

pytestmark = pytest.mark.gpu


def context(p, **env):
    os.environ.update(env)
    try:
        return Particles(p)
    finally:
        for k in env:
            os.environ.pop(k)


def lists(c):
    counts, ids = c.neighbors(stride=128)
    return [ids[i, :k].tolist() for i, k in enumerate(counts)], c.cells().tolist(), c.neighbor_stats()


@pytest.mark.parametrize("tile_min", ["1", "1000000000"])
@pytest.mark.parametrize("schedule", ["flat", "graph"])
def test_lists_after_a_reload_and_a_replay(tmp_path, schedule, tile_min):
    p = scene_params(0.1, 0.05, (0, 0, 0), (1, 1, 1), dt=0.005, max_neighbors=128)
    x = scenes.lattice_block(17, 17, 17, 0.05, (0.05, 0.05, 0.05))
    x = (x + np.random.default_rng(1).uniform(-1e-3, 1e-3, x.shape)).astype(np.float32)
    y = np.ascontiguousarray(x[::-1] * np.float32(0.9))
    with context(p, PBF_STEP_GRAPH="0", PBF_TILE_MIN="1000000000") as plain, \
            context(p, PBF_TILE_MIN=tile_min) as c:
        c.set_schedule(schedule)
        snap = str(tmp_path / "s.pbf")
        for k, state in enumerate((x, x, y, None)):
            for q in (plain, c):
                if state is None:
                    q.load_snapshot(snap)
                else:
                    q.load(state, None)
                # The lists of the state before the load are gone.
                with pytest.raises(PbfError):
                    q.neighbors(stride=128)
            for _ in range(3 if k == 0 else 1):
                plain.time_step()
                c.time_step()
            if k == 1:
                plain.save_snapshot(snap)
            assert lists(c) == lists(plain), k
