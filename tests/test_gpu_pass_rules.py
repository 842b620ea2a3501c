"""The step on both sides of the sizes where its passes change from a wave to a
quad per particle, as one scene and as two scenes of one context (which keep
their waves longer), bit for bit against the oracle."""
import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles

pytestmark = pytest.mark.gpu

BOX = (3.0, 3.0, 3.0)


def _scene(n, seed):
    k = int(np.ceil(n ** (1 / 3)))
    x = scenes.lattice_block(k, k, k, 0.05, (0.2, 0.2, 0.2))[:n]
    r = np.random.default_rng(seed)
    x = (x + r.uniform(-1e-3, 1e-3, x.shape)).astype(np.float32)
    return x, r.uniform(-0.3, 0.3, x.shape).astype(np.float32)


def _params():
    return scene_params(0.1, 0.05, (0, 0, 0), BOX, dt=0.005)


@pytest.mark.parametrize("n", [6144, 6145, 11264, 11265, 16384, 16385])
def test_one_scene(orc, n):
    p = _params()
    x, v = _scene(n, n)
    f = Particles(p)
    f.load(x, v)
    f.time_step(nsteps=3)
    gx, gv, _ = f.read()
    f.close()
    ox, ov, _ = orc.step(p, x, v, 3, orc.NBR_GRID)
    assert np.array_equal(gx.view(np.uint32), ox.view(np.uint32))
    assert np.array_equal(gv.view(np.uint32), ov.view(np.uint32))


@pytest.mark.parametrize("n", [6145, 11265, 12289, 16385])
def test_two_scenes(orc, n):
    p = _params()
    parts = [_scene(n // 3, n), _scene(n - n // 3, n + 1)]
    f = Particles(p, scenes=[(len(x), (0, 0, 0), BOX) for x, _ in parts])
    f.load(np.concatenate([x for x, _ in parts]), np.concatenate([v for _, v in parts]))
    f.time_step(nsteps=2)
    gx, gv, _ = f.read()
    f.close()
    o = 0
    for x, v in parts:
        ox, ov, _ = orc.step(p, x, v, 2, orc.NBR_GRID)
        assert np.array_equal(gx[o:o + len(x)].view(np.uint32), ox.view(np.uint32))
        assert np.array_equal(gv[o:o + len(x)].view(np.uint32), ov.view(np.uint32))
        o += len(x)
