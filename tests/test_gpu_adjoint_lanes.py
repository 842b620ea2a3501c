"""The adjoint's lists over 16, 4 or 1 lanes and its short divisions and
square roots, against one lane per particle with the compiler's divisions.

The sizes are a lone particle, a pair, partial waves, and both sides of the
16,384 particles up to which a particle has sixteen lanes.  An EPS_D below
2^-47 keeps the general sequences (no pair is that close, so nothing else
changes).  The splits add the same terms in other orders and a short quotient
may differ in its last bit: 1e-5 of the largest component, the bound the
lane splits keep among themselves.  The forward pass gives the same bits.
"""
import os

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.adjoint import Rollout

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _run(p, x, v, target, lanes=None):
    if lanes:
        os.environ["PBF_ADJ_LANES"] = lanes
    try:
        r = Rollout(p, len(x), 2, checkpoint_every=1)
    finally:
        os.environ.pop("PBF_ADJ_LANES", None)
    xT, _ = r.forward(x, v, p.k_tensile)
    xbar = ((2.0 / len(x)) * (xT.astype(np.float64) - target)).astype(np.float32)
    xb, vb, kb = r.backward(xbar)
    assert r.replay_mismatches() == 0
    r.close()
    return xT, xb, vb, kb


@pytest.mark.parametrize("n", [1, 2, 3, 63, 65, 1001, 16384, 16385])
def test_lanes_and_short_sequences(n):
    sc, target = scenes.diff_block(n_side=26 if n > 1331 else 11, steps=2)
    x, v, target = sc.x[:n], sc.v[:n], target[:n].astype(np.float64)
    ref = _run(sc.params.replace(eps_d=1e-15), x, v, target, "1")
    for lanes in (None, "16", "4"):
        out = _run(sc.params, x, v, target, lanes)
        assert np.array_equal(out[0].view(np.uint32), ref[0].view(np.uint32))
        for a, b in zip(out[1:3], ref[1:3]):
            assert np.isfinite(b).all() and np.abs(a - b).max() <= TOL * np.abs(b).max()
        assert abs(out[3] - ref[3]) <= TOL * abs(ref[3])


@pytest.mark.parametrize("iterations", [1, 2])
def test_few_iterations(orc, iterations):
    """The tape of one and two solver iterations (x*_0 in the sorted
    prediction, the last x* unpacked, 12-byte records between): dL/dv0 along
    itself against FP64 central differences of the oracle, within 1e-3."""
    sc, target = scenes.diff_block(n_side=8, steps=3)
    p = sc.params.replace(iterations=iterations)
    r = Rollout(p, sc.n, 3, checkpoint_every=2)
    xT, _ = r.forward(sc.x, sc.v, p.k_tensile)
    t64 = target.astype(np.float64)
    _, vb, _ = r.backward(((2.0 / sc.n) * (xT.astype(np.float64) - t64)).astype(np.float32))
    assert r.replay_mismatches() == 0 and r.stats()[1] == 0
    r.close()

    def loss(v):
        x, _, _ = orc.step(p.as_dict(), sc.x.astype(np.float64), v, 3, dtype=np.float64)
        return float(np.mean(np.sum((x - t64) ** 2, axis=1)))

    g = vb.astype(np.float64)
    gn = float(np.linalg.norm(g))
    v0, h = sc.v.astype(np.float64), 1e-6
    fd = (loss(v0 + h * g / gn) - loss(v0 - h * g / gn)) / (2 * h)
    assert abs(fd - gn) <= 1e-3 * abs(fd)
