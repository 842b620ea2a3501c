"""pbf_step_async does not wait for what is enqueued, also where a change of dt
replaces captured steps that queued calls still replay; many such changes in a
row, loads and density queries between, give the bits of plain launches."""
import os
import time

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.params import scene_params
from fluid_amd.pbf import Particles

pytestmark = pytest.mark.gpu


def _state(n):
    k = int(np.ceil(n ** (1 / 3)))
    r = np.random.default_rng(n)
    x = scenes.lattice_block(k, k, k, 0.05, (0.05, 0.05, 0.05))[:n]
    x = (x + r.uniform(-1e-3, 1e-3, x.shape)).astype(np.float32)
    box = 0.05 * k + 0.6
    return x, scene_params(0.1, 0.05, (0, 0, 0), (box,) * 3, dt=0.002, max_neighbors=256)


def _plain(p):
    os.environ["PBF_STEP_GRAPH"] = "0"
    try:
        return Particles(p)
    finally:
        os.environ.pop("PBF_STEP_GRAPH")


def test_a_change_of_dt_does_not_wait():
    x, p = _state(120000)
    with Particles(p) as c:
        c.set_schedule("graph")
        c.load(x, None)
        waited = []
        for _ in range(3):  # the first captures, and warms the runtime
            t0 = time.perf_counter()
            for k in range(3):
                c.step_async(100, dt=p.dt * (1.0 + 0.01 * (k % 2)))
            t1 = time.perf_counter()
            c.sync()
            waited.append((t1 - t0) / (time.perf_counter() - t0))
        # Waiting at each of the two changes would take two thirds of it.
        assert min(waited) < 0.5, waited


@pytest.mark.parametrize("n", [1000, 5000])
@pytest.mark.parametrize("schedule", ["flat", "graph"])
def test_changes_of_dt_in_flight(n, schedule):
    x, p = _state(n)
    with _plain(p) as a, Particles(p) as b:
        b.set_schedule(schedule)
        for c in (a, b):
            c.load(x, None)
        for part in range(3):
            for k in range(45):
                dt = p.dt * (1.0 + 0.01 * (k // (1 + part) % 5))
                for c in (a, b):
                    c.step_async((1, 3, 7, 12)[k % 4], dt=dt)
            if part == 1:
                rho = [c.estimate_densities() for c in (a, b)]
                assert np.array_equal(rho[0].view(np.uint32), rho[1].view(np.uint32))
            else:
                for c in (a, b):
                    c.sync()
            for u, w in zip(a.read(), b.read()):
                assert np.array_equal(u.view(np.uint32), w.view(np.uint32))
            if part == 1:
                for c in (a, b):
                    c.step_async(9)
                    c.load(x, None)
