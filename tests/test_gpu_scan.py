"""The cell scan at the edges of its 1,024-cell tiles and on both sides of the
4,096 tiles up to which the tile offsets are added up by the last launch, bit
for bit against the oracle (a wrong cell start sorts particles apart)."""
import os

import numpy as np
import pytest

from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (3, 11, 31), (16, 8, 8), (41, 5, 5), (32, 32, 4),
                                  (256, 128, 128), (257, 128, 128)])
def test_cell_starts_at_tile_edges(orc, dims):
    h = 0.1
    box = [(k - 0.5) * h for k in dims]
    p = scene_params(h, h / 2, (0, 0, 0), box, dt=0.005, max_neighbors=512)
    r = np.random.default_rng(sum(dims))
    # Both ends of the grid, and all of it.
    u = r.uniform(0.0, 1.0, (300, 3))
    lo, hi, side = np.zeros(3), np.array(box), np.minimum(np.array(box), 4 * h)
    x = np.concatenate([lo + side * u[:100], hi - side * u[100:200], hi * u[200:]])
    x = np.clip(x, lo, hi).astype(np.float32)
    x = np.minimum(x, np.array(box, np.float32))
    v = r.uniform(-0.5, 0.5, x.shape).astype(np.float32)
    os.environ["PBF_NO_SMALL_SORT"] = "1"
    try:
        f = Particles(p)
    finally:
        os.environ.pop("PBF_NO_SMALL_SORT", None)
    assert tuple(f.grid_dims()) == dims
    f.load(x, v)
    f.time_step(nsteps=2)
    gx, gv, _ = f.read()
    f.close()
    ox, ov, _ = orc.step(p, x, v, 2, orc.NBR_GRID)
    assert np.array_equal(gx.view(np.uint32), ox.view(np.uint32))
    assert np.array_equal(gv.view(np.uint32), ov.view(np.uint32))


@pytest.mark.parametrize("dims", [(1, 1, 1), (7, 5, 7), (32, 16, 16), (33, 16, 16), (32, 32, 32)])
@pytest.mark.parametrize("n", [1, 64, 1024, 1025, 2049, 3073, 4096, 4097])
def test_single_workgroup_sort(orc, dims, n):
    """The single-workgroup sort at one to four particles a thread and one
    particle beyond, with the cell starts in LDS (8,192 cells) and in global
    memory, many particles a cell."""
    h = 0.1
    box = [(k - 0.5) * h for k in dims]
    p = scene_params(h, h / 2, (0, 0, 0), box, dt=0.005, max_neighbors=1024)
    r = np.random.default_rng(n + sum(dims))
    # At most ~900 particles within h of one another.
    if dims == (1, 1, 1) and n > 900:
        pytest.skip("more neighbours than a list holds")
    x = (np.array(box) * r.uniform(0.0, 1.0, (n, 3))).astype(np.float32)
    x = np.minimum(x, np.array(box, np.float32))
    v = r.uniform(-0.5, 0.5, x.shape).astype(np.float32)
    f = Particles(p)
    f.load(x, v)
    f.time_step(nsteps=2)
    gx, gv, _ = f.read()
    f.close()
    ox, ov, _ = orc.step(p, x, v, 2, orc.NBR_GRID)
    assert np.array_equal(gx.view(np.uint32), ox.view(np.uint32))
    assert np.array_equal(gv.view(np.uint32), ov.view(np.uint32))
