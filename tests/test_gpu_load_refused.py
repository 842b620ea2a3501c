"""A refused first load leaves a context as it was created: no particles to
count, step or read, whichever side checks it, for one scene and for several."""
import numpy as np
import pytest

from fluid_amd._lib import lib
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles, PbfError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [100, 6000])
@pytest.mark.parametrize("scenes", [1, 3])
def test_refused_first_load(n, scenes):
    p = scene_params(0.1, 0.05, (0, 0, 0), (1, 1, 1))
    spec = None if scenes == 1 else [(n, (0, 0, 0), (1, 1, 1))] * scenes
    x = np.random.default_rng(1).uniform(0, 1, (n * scenes, 3)).astype(np.float32)
    bad = x.copy()
    bad[n * scenes - 1, 2] = np.nan
    with Particles(p, scenes=spec) as c:
        for _ in range(2):
            with pytest.raises(PbfError) as e:
                c.load(bad, None)
            assert e.value.code == -1 and f"particle {n * scenes - 1} " in str(e.value)
            assert lib().pbf_count(c._ctx) == 0
            with pytest.raises(PbfError) as e:
                c.time_step()
            assert e.value.code == -4
        c.load(x, None)
        assert lib().pbf_count(c._ctx) == n * scenes
        with pytest.raises(PbfError):
            c.load(bad, None)
        assert lib().pbf_count(c._ctx) == n * scenes
        assert np.array_equal(c.read()[0], x)
