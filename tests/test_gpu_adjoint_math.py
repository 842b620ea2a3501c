"""The adjoint's short square root, reciprocal, divisions and quotients round as
the IEEE operations do: gradients with them and without (PBF_IEEE_MATH=1) have
the same bits, over smoothing lengths and cut-offs EPS_D, with pairs at many
distances and one closer than EPS_D."""
import os

import numpy as np
import pytest

from fluid_amd.adjoint import Rollout
from fluid_amd.params import EPS_D, scene_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,eps_d", [(0.1, EPS_D), (0.3, EPS_D), (0.02, EPS_D), (1.0, 1e-6),
                                     (0.1, 2e-12), (0.1, 1e-13)])
def test_gradients_with_the_short_sequences_have_the_same_bits(h, eps_d):
    p = scene_params(h, h / 2, (-1,) * 3, (20 * h,) * 3, dt=0.005, max_neighbors=256)
    p = p.replace(eps_d=eps_d)
    r = np.random.default_rng(5)
    x = (h * r.uniform(0, 5, (900, 3))).astype(np.float32)
    x[0], x[1] = 0.0, (1e-12, 0.0, 0.0)
    x[3] = x[2]
    v = r.uniform(-h, h, x.shape).astype(np.float32)
    xb = r.uniform(-1, 1, x.shape).astype(np.float32)
    vb = r.uniform(-1, 1, x.shape).astype(np.float32)
    out = []
    for ieee in (False, True):
        if ieee:
            os.environ["PBF_IEEE_MATH"] = "1"
        try:
            f = Rollout(p, len(x), 2, 1)
        finally:
            os.environ.pop("PBF_IEEE_MATH", None)
        f.forward(x, v, p.k_tensile)
        out.append(f.backward(xb, vb))
    for a, b in zip(out[0][:2], out[1][:2]):
        assert np.isfinite(a).all()
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert out[0][2] == out[1][2]
