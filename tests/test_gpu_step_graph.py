"""Calls of several steps of a small state replay four captured steps at a time
once the same dt comes twice: every call equals plain launches
(PBF_STEP_GRAPH=0) bit for bit, over calls one step below, at and beyond the
shortest that replays, remainders of 0 to 3 steps, one-step calls, reads, a
reload and changes of dt between, asynchronous calls with a change of dt while
replays are queued, and the graph schedule; the first 12 steps against the
oracle."""
import os

import numpy as np
import pytest

from fluid_amd import scenes
from fluid_amd.pbf import Particles

pytestmark = pytest.mark.gpu


def _ctx(p, x, v, env=None, schedule=None):
    old = os.environ.get("PBF_STEP_GRAPH")
    if env is not None:
        os.environ["PBF_STEP_GRAPH"] = env
    try:
        c = Particles(p)
    finally:
        if env is not None:
            os.environ.pop("PBF_STEP_GRAPH", None)
            if old is not None:
                os.environ["PBF_STEP_GRAPH"] = old
    if schedule:
        c.set_schedule(schedule)
    c.load(x, v)
    return c


def _same(a, b):
    return all(np.array_equal(u.view(np.uint32), w.view(np.uint32)) for u, w in zip(a, b))


@pytest.mark.parametrize("side", [8, 20, 22])
def test_replays_equal_plain_launches(orc, side):
    sc, _ = scenes.diff_block(n_side=side, steps=1)
    p = sc.params
    plain = _ctx(p, sc.x, sc.v, env="0")
    flat, graph = _ctx(p, sc.x, sc.v), _ctx(p, sc.x, sc.v, schedule="graph")
    done = 0
    for k, n in enumerate((6, 6, 5, 7, 1, 8, 9, 10, 13, 6, 6, 2, 18)):
        dt = None if k < 9 else 0.5 * p.dt
        if k == 7:
            for c in (plain, flat, graph):
                c.load(sc.x, sc.v)
        for c in (plain, flat, graph):
            c.time_step(dt=dt, nsteps=n)
        ref = plain.read()
        assert _same(ref, flat.read()) and _same(ref, graph.read()), (k, n)
        done += n
        if done == 12:
            ox, ov, _ = orc.step(p, sc.x, sc.v, 12, orc.NBR_GRID)
            assert _same(ref[:2], (ox, ov))
    for c in (plain, flat, graph):
        c.load(sc.x, sc.v)
        for dt, n in ((p.dt, 14), (p.dt, 14), (0.5 * p.dt, 6), (0.5 * p.dt, 14), (p.dt, 6)):
            c.step_async(n, dt=dt)
        c.sync()
    ref = plain.read()
    assert _same(ref, flat.read()) and _same(ref, graph.read())
    for c in (plain, flat, graph):
        c.close()


def test_buffer_swaps_between_calls():
    """Densities and a density lattice between the calls swap the state's
    buffers under the captured steps."""
    sc, _ = scenes.diff_block(n_side=10, steps=1)
    plain, flat = _ctx(sc.params, sc.x, sc.v, env="0"), _ctx(sc.params, sc.x, sc.v)
    graph = _ctx(sc.params, sc.x, sc.v, schedule="graph")
    for k, n in enumerate((7, 7, 7, 10, 1, 1, 1, 6, 6, 6)):
        out = []
        for c in (plain, flat, graph):
            c.time_step(nsteps=n)
            rho = c.estimate_densities() if k in (1, 3, 5, 7) else np.zeros(1, np.float32)
            if k in (2, 7):
                p = sc.params
                rho = c.density_lattice(p.box_lo, p.box_hi, 0.5, (4, 4, 4))
            out.append((np.ascontiguousarray(rho, np.float32), *c.read()))
        assert _same(out[0], out[1]) and _same(out[0], out[2]), (k, n)
    for c in (plain, flat, graph):
        c.close()
