"""The scaled short division by h^9 over smoothing lengths: in use down to
h = 0.002, and everywhere (also where no scale fits, or the general division
stays) two steps with the bits of the IEEE sequences (PBF_IEEE_MATH=1)."""
import os

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h", [2000.0, 100.0, 1.0, 0.3, 0.1, 0.03, 0.02, 0.01, 0.002, 0.001])
def test_division_over_smoothing_lengths(h):
    p = scene_params(h, h / 2, (0, 0, 0), (12 * h, 12 * h, 12 * h), dt=0.005)
    x = scenes.lattice_block(11, 11, 11, h / 2, (h, h, h))
    r = np.random.default_rng(7)
    x = (x + r.uniform(-0.1 * h, 0.1 * h, x.shape)).astype(np.float32)
    v = r.uniform(-h, h, x.shape).astype(np.float32)
    out = []
    for ieee in (False, True):
        if ieee:
            os.environ["PBF_IEEE_MATH"] = "1"
        try:
            f = Particles(p)
        finally:
            os.environ.pop("PBF_IEEE_MATH", None)
        if ieee:
            assert not f.math_flags()["div"]
        elif 0.002 <= h <= 1.0:
            assert f.math_flags()["div"]
        f.load(x, v)
        rho = f.estimate_densities()
        f.time_step(nsteps=2)
        out.append((rho, *f.read()))
        f.close()
    for a, b in zip(*out):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
