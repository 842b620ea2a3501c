"""Constants with which a particle's own lambda, tensile scale or velocity is
infinite, or which put clamped positions far outside the box: the padding
entries of the tiles' lists must add nothing there, so states that would step
on tiles (PBF_TILE_MIN=1) give what the per-lane passes give."""
import os

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles

pytestmark = pytest.mark.gpu

CASES = {
    "plain": {},
    "tensile_scale_infinite": {"dq": 1.0, "iterations": 1},
    "no_relaxation": {"epsilon": 0.0, "rest_density": 1e25, "iterations": 2},
    "velocity_infinite": {"dt": 1e-39, "iterations": 1},
    "velocity_overflows": {"dt": 1e-38, "iterations": 3},
    "clamped_beyond_the_padding": {"eps_d": 1.4},
}


@pytest.mark.parametrize("name", list(CASES))
def test_padding_adds_nothing(name):
    p = scene_params(0.1, 0.05, (0, 0, 0), (1, 1, 1), dt=0.005, max_neighbors=128)
    p = p.replace(**CASES[name])
    x = scenes.lattice_block(9, 9, 9, 0.05, (0.3, 0.3, 0.3))
    r = np.random.default_rng(4)
    x = (x + r.uniform(-1e-3, 1e-3, x.shape)).astype(np.float32)
    v = r.uniform(-0.5, 0.5, x.shape).astype(np.float32)
    out = []
    for tile_min in ("1", "1000000000"):
        os.environ.update(PBF_TILE_MIN=tile_min, PBF_NO_SMALL_SORT="1", PBF_WIDE_MAX="0",
                          PBF_QUAD_MAX="0")
        try:
            c = Particles(p)
        finally:
            for k in ("PBF_TILE_MIN", "PBF_NO_SMALL_SORT", "PBF_WIDE_MAX", "PBF_QUAD_MAX"):
                os.environ.pop(k)
        with c:
            c.load(x, v)
            c.time_step(nsteps=1)
            out.append(c.read())
    for a, b in zip(*out):
        # Bit for bit but for the payload of NaN.
        assert np.array_equal(np.isnan(a), np.isnan(b))
        a, b = np.nan_to_num(a, nan=1.0), np.nan_to_num(b, nan=1.0)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
