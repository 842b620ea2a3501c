"""What the framework is timed on: passes of its public entry points over the
range of states that its users step.

Every case is a dict of plain values; ``prepare`` makes its inputs from a seed
and the handle that a program keeps, ``run`` makes one pass.  A pass that
simulates starts from the loaded initial state, so that every pass does the
same work: load, steps, read, as the ``-p``/``-d`` path of the reference does
(src/application.cpp:302-344, src/pathtracer.cpp:444-480).

Kinds:

* ``native``   the reference's own scenes at its native constants (h 0.3, 12
  iterations, the Cornell box): a lattice of a few hundred to a few thousand
  particles.  ``frames`` > 0 makes one call per step with a read after each,
  as its viewer does; else one call of ``steps`` steps.
* ``dam``      a lattice block collapsing in a box three times as long.
* ``spheres``  two lattice spheres thrown at each other, then the floor.
* ``mesh``     a dam over a triangle-mesh sphere in a triangle-mesh box.
* ``batch``    many scenes of uneven sizes in one context.
* ``adjoint``  a differentiable rollout, forward and backward.
* ``surface``  load-time densities and the marching-cubes corner lattice.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch
import torch.utils.checkpoint

from fluid_amd import mesh as meshes
from fluid_amd.adjoint import Rollout
from fluid_amd.params import reference_params, scene_params
from fluid_amd.pbf import Particles


def listed():
    return [
        # The reference's particles/p.xml (720 particles) for one simulated
        # second, 63 steps of 16 ms in one call: launches and latency.
        {"name": "native_720_second", "kind": "native", "n": 720, "spacing": 0.15, "steps": 63,
         "frames": 0},
        # The size of particles/spheres_p.xml in the viewer's loop: one
        # timeStep() and one read of the positions per frame.
        {"name": "native_2106_frames", "kind": "native", "n": 2106, "spacing": 0.1, "steps": 1,
         "frames": 24},
        # An interactive-size dam with a ragged count.
        {"name": "dam_20011", "kind": "dam", "n": 20011, "steps": 40},
        # A mid-size dam, between the smallest states and those that fill the
        # card.
        {"name": "dam_70001", "kind": "dam", "n": 70001, "steps": 40},
        # The dam break: its column keeps compressing over 200 steps, from 28
        # neighbours to about 98 on average.
        {"name": "dam_break_262144", "kind": "dam", "n": 262144, "steps": 200},
        # A mesh collider in a dam that fills the card.
        {"name": "mesh_300007", "kind": "mesh", "n": 300007, "steps": 20},
        # Two steps of a million particles, ragged: the large state at rest
        # density, with the load and the read that a short call pays for.
        {"name": "spheres_1000003", "kind": "spheres", "n": 1000003, "steps": 2},
        # The largest scene over its whole run, through both impacts.
        {"name": "two_spheres_4096000", "kind": "spheres", "n": 4096000, "steps": 100},
        # Uneven small scenes stepped together.
        {"name": "batch_128", "kind": "batch", "scenes": 128, "lo": 1000, "hi": 32768,
         "steps": 20},
        # Gradients of a short rollout of a small state and of the mid-size
        # block that the gradient workload uses.
        {"name": "adjoint_1000", "kind": "adjoint", "n": 1000, "steps": 10, "every": 4},
        {"name": "adjoint_32768", "kind": "adjoint", "n": 32768, "steps": 10, "every": 5},
        # Surface extraction's inputs for a loaded state.
        {"name": "surface_500009", "kind": "surface", "n": 500009, "step": 0.5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["native", "dam", "dam", "dam", "spheres", "spheres", "mesh", "batch",
                       "adjoint", "surface"])
    if kind == "native":
        spacing = rng.choice([0.1, 0.15])
        n = _log_int(rng, 200, 4000 if spacing == 0.1 else 1500)
        if rng.random() < 0.5:
            return {"kind": kind, "n": n, "spacing": spacing, "steps": 1,
                    "frames": rng.randint(4, 40)}
        return {"kind": kind, "n": n, "spacing": spacing, "steps": rng.randint(10, 80),
                "frames": 0}
    if kind == "dam":
        n = _log_int(rng, 3000, 400000)
        return {"kind": kind, "n": n, "steps": rng.randint(2, 120)}
    if kind == "spheres":
        n = _log_int(rng, 100000, 4000000)
        return {"kind": kind, "n": n, "steps": _log_int(rng, 2, 60)}
    if kind == "mesh":
        n = _log_int(rng, 5000, 1000000)
        return {"kind": kind, "n": n, "steps": rng.randint(4, 40)}
    if kind == "batch":
        lo = _log_int(rng, 500, 2000)
        return {"kind": kind, "scenes": _log_int(rng, 8, 256), "lo": lo,
                "hi": _log_int(rng, 8000, 32768), "steps": rng.randint(4, 30)}
    if kind == "adjoint":
        return {"kind": kind, "n": _log_int(rng, 500, 100000), "steps": rng.randint(2, 10),
                "every": rng.randint(2, 8)}
    return {"kind": "surface", "n": _log_int(rng, 5000, 2000000),
            "step": rng.choice([0.5, 0.75, 1.0])}


# ------------------------------------------------------------- inputs --


def _uniform(seed, shape, amp):
    g = torch.Generator().manual_seed(int(seed))
    return (torch.rand(shape, generator=g, dtype=torch.float64) * 2.0 - 1.0).numpy() * amp


def _block(n, side_x, side_z, spacing, corner):
    """The first n points of a lattice of side_x * side_z columns, in layers
    from the floor up."""
    q = np.arange(n)
    i, k, j = q % side_x, (q // side_x) % side_z, q // (side_x * side_z)
    return np.asarray(corner, np.float64) + spacing * np.stack([i, j, k], axis=1)


@functools.lru_cache(maxsize=2)
def _ball(n):
    """The n points of the unit lattice nearest to the origin."""
    r = int(math.ceil((3.0 * n / (4.0 * math.pi)) ** (1.0 / 3.0))) + 2
    a = np.arange(-r, r + 1)
    k, j, i = np.meshgrid(a, a, a, indexing="ij")
    r2 = (i * i + j * j + k * k).ravel()
    cut = np.partition(r2, n - 1)[n - 1]
    sel = np.nonzero(r2 < cut)[0]
    sel = np.concatenate([sel, np.nonzero(r2 == cut)[0][: n - len(sel)]])
    return np.stack([i.ravel()[sel], j.ravel()[sel], k.ravel()[sel]], axis=1).astype(np.float64)


def _scene(case):
    """(lattice points, velocities, jitter amplitude, params) of a case with
    one scene."""
    kind, n = case["kind"], case["n"]
    if kind == "native":
        s = case["spacing"]
        side = 19 if s == 0.1 else 12
        base = _block(n, side, side, s, (-0.9, 0.1, -0.9))
        vel = np.zeros_like(base)
        vel[:, 1] = -1.0 if s == 0.1 else -0.01
        p = reference_params().replace(rest_density=700.0 if s == 0.1 else 150.0)
        return base, vel, 1e-3, p
    if kind == "adjoint":
        side = max(2, int(round(n ** (1.0 / 3.0))))
        s = 0.05
        base = _block(n, side, side, s, (-0.5 * s * (side - 1), 0.0, -0.5 * s * (side - 1)))
        p = scene_params(0.1, s, (-6, -6, -6), (6, 6, 6), dt=0.01)
        return base, np.zeros_like(base), 1e-3, p
    if kind == "spheres" or kind == "surface":
        a = n // 2
        b = n - a
        s = 0.8 * (4.0 * math.pi / 3.0 / max(a, 1)) ** (1.0 / 3.0)
        base = np.concatenate([np.array([1.2, 1.5, 1.5]) + s * _ball(b)[:a],
                               np.array([3.8, 1.5, 1.5]) + s * _ball(b)])
        vel = np.zeros_like(base)
        vel[:a, 0], vel[a:, 0] = 2.0, -2.0
        p = scene_params(2 * s, s, (0, 0, 0), (5, 3, 3), dt=0.005, max_neighbors=512)
        return base, vel, 0.0156 * s, p
    # dam, mesh
    side = max(2, int(math.ceil(n ** (1.0 / 3.0) - 1e-9)))
    L = 0.8 if n <= 8192 else 1.6
    s = L / side
    base = _block(n, side, side, s, (s / 2, s / 2, s / 2))
    p = scene_params(2 * s, s, (0, 0, 0), (3 * L, 1.875 * L, L), dt=0.01 if s >= 0.025 else 0.005,
                     max_neighbors=1024 if kind == "mesh" else 2048)
    return base, np.zeros_like(base), 0.02 * s, p


def _inputs(case, seed):
    base, vel, amp, p = _scene(case)
    x = (base + _uniform(seed, base.shape, amp)).astype(np.float32)
    v = (vel + _uniform(seed + 7919, base.shape, 1e-2)).astype(np.float32)
    x = np.clip(x, np.asarray(p.box_lo, np.float32), np.asarray(p.box_hi, np.float32))
    return x, v, p


def _batch_inputs(case, seed):
    """The sizes and boxes of the scenes come from the case, their jitter and
    velocities from the seed."""
    rng = np.random.default_rng(case["scenes"] * 7 + case["lo"])
    counts = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]),
                                size=case["scenes"])).astype(np.int64)
    s, h = 0.05, 0.1
    xs, vs, spec = [], [], []
    vel = _uniform(seed + 7919, (len(counts), 3), 1.0)
    for q, c in enumerate(counts):
        c = int(c)
        side = int(math.ceil(c ** (1.0 / 3.0)))
        if rng.uniform() < 0.5:
            pts = _block(c, side, side, s, (s / 2, s / 2, s / 2))
            box = np.array([side * s * 2, side * s * 1.5, side * s])
        else:
            rad = s * (3.0 * c / (4.0 * math.pi)) ** (1.0 / 3.0) + s
            box = np.full(3, 2.5 * rad)
            pts = box / 2 + s * _ball(c)
        spec.append((c, (0.0, 0.0, 0.0), tuple(float(t) for t in box)))
        xs.append(pts)
        vs.append(np.broadcast_to(vel[q], pts.shape))
    x = np.concatenate(xs)
    x = (x + _uniform(seed, x.shape, 1e-3)).astype(np.float32)
    return x, np.concatenate(vs).astype(np.float32), spec, scene_params(h, s, (0, 0, 0), (1, 1, 1))


def _lattice(case, p):
    step = float(np.float32(case["step"] * p.h))
    counts = [int((hi - lo) / step) + 2 for lo, hi in zip(p.box_lo, p.box_hi)]
    return step, counts


# -------------------------------------------------------------- passes --


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "batch":
        x, v, spec, p = _batch_inputs(case, seed)
        st["handle"] = Particles(p, scenes=spec)
    else:
        x, v, p = _inputs(case, seed)
        if kind == "adjoint":
            st["handle"] = Rollout(p, case["n"], case["steps"], case["every"])
            st["target"] = (x + np.array([0.5, 0.0, 0.3])
                            + _uniform(seed + 104729, x.shape, 1e-3)).astype(np.float32)
        else:
            st["handle"] = Particles(p)
        if kind == "mesh":
            st["handle"].set_mesh(*_mesh(p))
        if kind == "surface":
            st["lattice"] = _lattice(case, p)
    st.update(x=x, v=v, params=p)
    return st


def _mesh(p):
    lo, hi = np.asarray(p.box_lo), np.asarray(p.box_hi)
    ball = meshes.icosphere((0.55 * hi[0], 0.1 * hi[1], 0.5 * hi[2]), 0.15 * hi[2], subdiv=4)
    pos, nrm, tri = meshes.merge(meshes.box(lo, hi), ball)
    return pos, nrm, tri, meshes.default_skin(pos, lo, hi)


def run(st):
    case, h = st["case"], st["handle"]
    kind = case["kind"]
    if kind == "adjoint":
        x, v = h.forward(st["x"], st["v"], st["params"].k_tensile)
        gx = (x - st["target"]) * np.float32(2.0 / case["n"])
        xb, vb, kb = h.backward(gx)
        return {"x": x, "v": v, "dx0": xb, "dv0": vb, "dk": kb}
    h.load(st["x"], st["v"])
    if kind == "surface":
        rho = h.estimate_densities()
        step, counts = st["lattice"]
        p = st["params"]
        return {"rho": rho, "field": h.density_lattice(p.box_lo, p.box_hi, step, counts)}
    if kind == "native" and case["frames"]:
        for _ in range(case["frames"]):
            h.time_step()
            out = h.read()
    else:
        h.time_step(nsteps=case["steps"])
        out = h.read()
    return {"x": out[0], "v": out[1], "rho": out[2]}


# Neighbours of a particle at rest, and arithmetic of one pair: the distance
# and both kernels, about 40 operations a pass.
def _pair_flops(n, passes, neighbours):
    return float(n) * passes * neighbours * 40.0


def work(case):
    kind = case["kind"]
    if kind == "batch":
        rng = np.random.default_rng(case["scenes"] * 7 + case["lo"])
        n = int(np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]),
                                   size=case["scenes"])).astype(np.int64).sum())
        return {"bytes": 52.0 * n, "flops": case["steps"] * _pair_flops(n, 11, 28)}
    n = case["n"]
    if kind == "native":
        steps = case["frames"] or case["steps"]
        return {"bytes": 24.0 * n + 28.0 * n * max(1, case["frames"]),
                "flops": steps * _pair_flops(n, 27, 75 if case["spacing"] == 0.1 else 22)}
    if kind == "adjoint":
        # Forward, and its adjoint at about twice the arithmetic.
        return {"bytes": 84.0 * n, "flops": 3.0 * case["steps"] * _pair_flops(n, 11, 28)}
    if kind == "surface":
        _, counts = _lattice(case, _scene(case)[3])
        m = int(np.prod(np.array(counts, dtype=np.int64)))
        pairs = n * (4.19 / case["step"] ** 3 + 33)
        return {"bytes": 24.0 * n + 4.0 * n + 4.0 * m, "flops": pairs * 15.0}
    return {"bytes": 52.0 * n, "flops": case["steps"] * _pair_flops(n, 11, 28)}


# ------------------------------------------------------- 64-bit results --


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _pairs(x, h2):
    """All ordered pairs (i, j), i != j, with |x_i - x_j|^2 <= h2."""
    cell = math.sqrt(h2) * 1.0001
    lo = x.min(0).values
    c = torch.floor((x - lo) / cell).long()
    dims = c.max(0).values + 3
    lin = ((c[:, 2] + 1) * dims[1] + c[:, 1] + 1) * dims[0] + c[:, 0] + 1
    keys, order = torch.sort(lin)
    ii, jj = [], []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            first = lin + (dz * dims[1] + dy) * dims[0] - 1
            s = torch.searchsorted(keys, first)
            e = torch.searchsorted(keys, first + 3)
            cnt = e - s
            i = torch.repeat_interleave(torch.arange(len(x), device=x.device), cnt)
            off = torch.arange(len(i), device=x.device) - torch.repeat_interleave(
                torch.cumsum(cnt, 0) - cnt, cnt)
            j = order[s[i] + off]
            keep = (i != j) & (((x[i] - x[j]) ** 2).sum(1) <= h2)
            ii.append(i[keep])
            jj.append(j[keep])
    return torch.cat(ii), torch.cat(jj)


class _Exact:
    """One step of the method in 64 bits (src/particles.cpp:250-297), for
    states that no wall touches."""

    def __init__(self, p):
        f = lambda t: float(np.float32(t))  # noqa: E731
        self.p, self.h = p, f(p.h)
        self.c1, self.c2 = f(p.poly6_coef), f(p.spiky_coef)
        self.rho0, self.eps, self.k = f(p.rest_density), f(p.epsilon), f(p.k_tensile)
        self.xc, self.dt, self.g = f(p.xsph_c), f(p.dt), f(p.gravity)
        self.dtv = self.dt * f(p.vort_eps)
        z = f(p.dq) * self.h
        self.S = self.h ** 9 / (self.c1 * (self.h ** 2 - z * z) ** 3)

    def kernels(self, x, i, j):
        r = x[i] - x[j]
        r2 = (r * r).sum(1)
        near = r2 < self.h ** 2
        t = torch.where(near, self.h ** 2 - r2, torch.zeros_like(r2))
        w = self.c1 * t ** 3 / self.h ** 9
        ok = near & (r2 > 1e-22)
        rl = torch.sqrt(torch.where(ok, r2, torch.ones_like(r2)))
        co = torch.where(ok, -3.0 * self.c2 * (self.h - rl) ** 2 / (self.h ** 6 * rl),
                         torch.zeros_like(rl))
        return w, co[:, None] * r

    def step(self, x, v, k):
        n = len(x)
        add = lambda i, q: torch.zeros((n,) + q.shape[1:], dtype=q.dtype,  # noqa: E731
                                       device=q.device).index_add(0, i, q)
        fall = torch.zeros(3, dtype=x.dtype, device=x.device)
        fall[1] = self.g * self.dt
        xs = x + (v - fall) * self.dt
        with torch.no_grad():
            i, j = _pairs(xs, self.h ** 2)
        for _ in range(self.p.iterations):
            w, g = self.kernels(xs, i, j)
            gs = g / self.rho0
            d = add(i, (gs * gs).sum(1)) + (add(i, gs) ** 2).sum(1)
            lam = -(add(i, w) / self.rho0 - 1.0) / (d + self.eps)
            s = -k * (w * self.S) ** self.p.n_tensile
            xs = xs + add(i, (lam[i] + lam[j] + s)[:, None] * g) / self.rho0
        v = (xs - x) / self.dt
        w, g = self.kernels(xs, i, j)
        u = v[j] - v[i]
        om = add(i, torch.linalg.cross(u, g))
        vx = v + self.xc * add(i, u * w[:, None])
        om2 = (om * om).sum(1)
        wn = torch.where(om2 > 0, torch.sqrt(torch.where(om2 > 0, om2, torch.ones_like(om2))), om2)
        eta = add(i, wn[j][:, None] * g)
        e2 = (eta * eta).sum(1)
        ok = e2 > 1e-22
        nrm = eta / torch.sqrt(torch.where(ok, e2, torch.ones_like(e2)))[:, None]
        turn = torch.where(ok[:, None], torch.linalg.cross(nrm, om), torch.zeros_like(om))
        return xs, vx + self.dtv * turn, add(i, w)


def exact(case, seed):
    kind, dev = case["kind"], _dev()
    if kind in ("dam", "spheres"):
        # Later states are chaotic: a 64-bit trajectory is another one.
        if case["steps"] > 2 or case["n"] > 2_000_000:
            return None
        x, v, p = _inputs(case, seed)
        e = _Exact(p)
        x, v = (torch.from_numpy(t).to(dev).double() for t in (x, v))
        with torch.no_grad():
            for _ in range(case["steps"]):
                x, v, rho = e.step(x, v, e.k)
        return {"x": x.cpu(), "v": v.cpu(), "rho": rho.cpu()}
    if kind == "adjoint":
        x, v, p = _inputs(case, seed)
        target = (x + np.array([0.5, 0.0, 0.3])
                  + _uniform(seed + 104729, x.shape, 1e-3)).astype(np.float32)
        e = _Exact(p)
        x0, v0, tg = (torch.from_numpy(t).to(dev).double() for t in (x, v, target))
        k = torch.tensor(e.k, dtype=torch.float64, device=dev, requires_grad=True)
        x0.requires_grad_(True)
        v0.requires_grad_(True)
        a, b = x0, v0
        for _ in range(case["steps"]):
            a, b = torch.utils.checkpoint.checkpoint(
                lambda s, t, q: e.step(s, t, q)[:2], a, b, k, use_reentrant=False)
        gx = (a.detach() - tg) * (2.0 / case["n"])
        a.backward(gx)
        return {"x": a.detach().cpu(), "v": b.detach().cpu(), "dx0": x0.grad.cpu(),
                "dv0": v0.grad.cpu(), "dk": float(k.grad)}
    if kind == "surface":
        x, _, p = _inputs(case, seed)
        e = _Exact(p)
        x = torch.from_numpy(x).to(dev).double()
        i, j = _pairs(x, e.h ** 2)
        rho = torch.zeros(len(x), dtype=x.dtype, device=dev).index_add(
            0, i, e.kernels(x, i, j)[0]) + e.c1 / e.h ** 3
        step, counts = _lattice(case, p)
        ax = []
        for a in range(3):
            q = np.float32(p.box_lo[a]) + np.arange(counts[a], dtype=np.float32) * np.float32(step)
            ax.append(torch.from_numpy(np.minimum(np.float32(p.box_hi[a]), q)).to(dev).double())
        base = torch.floor((x - torch.tensor(p.box_lo, device=dev)) / step).long()
        field = torch.zeros(counts[2] * counts[1] * counts[0], dtype=x.dtype, device=dev)
        span = int(math.ceil(1.0 / case["step"])) + 1
        for oz in range(-span, span + 1):
            for oy in range(-span, span + 1):
                for ox in range(-span, span + 1):
                    q = base + torch.tensor([ox, oy, oz], device=dev)
                    ok = ((q >= 0) & (q < torch.tensor(counts, device=dev))).all(1)
                    q, y = q[ok], x[ok]
                    r2 = sum((ax[a][q[:, a]] - y[:, a]) ** 2 for a in range(3))
                    t = (e.h ** 2 - r2).clamp(min=0.0)
                    field.index_add_(0, (q[:, 2] * counts[1] + q[:, 1]) * counts[0] + q[:, 0],
                                     e.c1 * t ** 3 / e.h ** 9)
        return {"rho": rho.cpu(), "field": field.reshape(counts[2], counts[1], counts[0]).cpu()}
    return None
