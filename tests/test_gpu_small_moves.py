"""Delta-p moves whose length rounds to zero: with EPS_D at or near 0 the
particle stays (the length is compared, not its components), bit for bit
against the oracle, from a particle at coordinate 0, where every float move
would show."""
import numpy as np
import pytest

from fluid_amd.params import Params
from fluid_amd.pbf import Particles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eps_d", [0.0, 1e-30, 1e-22])
@pytest.mark.parametrize("spiky", [1e-26, 2.5e-24, 1e-20, 1e-17, 1e-9])
def test_tiny_moves_bit_exact(orc, eps_d, spiky):
    p = Params().replace(gravity=0.0, eps_d=eps_d, spiky_coef=spiky, box_lo=(-1, -1, -1),
                         box_hi=(1, 1, 1))
    x = np.array([[0.0, 0.5, 0.5], [0.2, 0.5, 0.5], [0.0, 0.0, 0.0], [0.1, 0.1, 0.1]], np.float32)
    with Particles(p) as c:
        c.load(x, None)
        c.time_step(nsteps=2)
        gx, gv, grho = c.read()
    ox, ov, orho = orc.step(p, x, np.zeros_like(x), 2, orc.NBR_GRID)
    for a, b in ((gx, ox), (gv, ov), (grho, orho)):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
