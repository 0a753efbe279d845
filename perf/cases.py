"""Measured work: what a user of this framework has it do, through Solver,
Adjoint and MeshParticle.

A case is a dict of plain values; its "kind" names the work:

  roll      one particle rolling on a plane (the smallest system: launches and
            latency, 1e5 such steps make a run)
  cluster   a few hundred centimetre bodies with live rotation, colliding with
            one another, the floor and across the periodic faces
  packing   one packing of a parameter calibration (500..20000 millimetre
            particles, periodic in x and y, bottom layer on the floor)
  batch     many such packings in one solver
  pour      the large periodic lattice poured onto a floor
  bed       the same lattice compressed until its layers touch: the
            particle-particle narrow phase under load
  flow      the lattice with random velocities: bodies cross the periodic faces
            all the time, and the lists are built every few steps
  beam      a bonded face-centred cubic beam with a driven tip
  column    a packed column on a rough floor (fixed bodies), open sides
  adjoint   forward with checkpoints and reverse sweep of that column
  mesh      level-set grid of a closed triangle mesh

A pass of the stepping kinds advances `steps` steps and reads the state back,
as a program does between two output frames; "precision" is the state storage
("fp32" the production build, "fp64" the reference's). Particle templates are
the families the workloads use (their shapes are fixed, as a user's are);
positions, orientations, velocities and shape assignments come from the seed.
"""
from __future__ import annotations

import dataclasses
import functools
import math

import numpy as np
import torch

from fundem_amd import Adjoint, Solver
from fundem_amd import generators as G
from fundem_amd import workloads as W


def listed():
    return [
        # configuration 1 of the workloads: a single 2000-node body, 1e5 steps
        dict(name="roll", kind="roll", nodes=2000, steps=200, precision="fp32"),
        # parity-sized cluster with spin, the smallest many-body system
        dict(name="cluster-216", kind="cluster", n=216, steps=200, precision="fp32"),
        # one calibration run at the small end, in the all-FP64 build
        dict(name="packing-1500-fp64", kind="packing", n=1500, steps=100, precision="fp64"),
        # one calibration run at the large end
        dict(name="packing-16000", kind="packing", n=16000, steps=200, precision="fp32"),
        # a calibration sweep: log-uniform 500..20000 particles per packing
        dict(name="batch-64", kind="batch", count=64, lo=500, hi=20000, steps=100, precision="fp32"),
        # the headline: one million particles
        dict(name="pour-1000000", kind="pour", nx=100, ny=100, nz=100, steps=500, precision="fp32"),
        # contact-dense bed, every particle touching its neighbours above and below
        dict(name="bed-262144", kind="bed", nx=64, ny=64, nz=64, steps=50, precision="fp32"),
        # agitated particles: many list builds
        dict(name="flow-110592", kind="flow", nx=48, ny=48, nz=48, steps=200, precision="fp32"),
        # bonds: about six per body
        dict(name="beam-8192", kind="beam", nx=32, ny=8, nz=8, steps=500, precision="fp32"),
        # the differentiated configuration, forward only
        dict(name="column-4352", kind="column", nx=8, ny=8, nz=64, floor=16, steps=200, precision="fp32"),
        # and with its reverse sweep
        dict(name="adjoint-4352", kind="adjoint", nx=8, ny=8, nz=64, floor=16, steps=100, every=25,
             precision="fp32"),
        # mesh particle of about 5000 triangles at the default resolution
        dict(name="mesh-5120", kind="mesh", nu=80, nv=32, resolution=50),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["roll", "cluster", "packing", "batch", "pour", "bed", "flow", "beam", "column",
                       "adjoint", "mesh"])
    c = dict(kind=kind, precision=rng.choice(["fp32", "fp32", "fp64"]))
    if kind == "roll":
        c.update(nodes=log_int(200, 2000), steps=rng.randint(50, 200))
    elif kind == "cluster":
        c.update(n=log_int(8, 600), steps=rng.randint(150, 250))
    elif kind == "packing":
        c.update(n=log_int(500, 20000), steps=rng.randint(50, 200))
    elif kind == "batch":
        lo = log_int(500, 2000)
        c.update(count=rng.randint(3, 48), lo=lo, hi=log_int(lo, 20000), steps=rng.randint(30, 100))
    elif kind == "pour":
        c.update(nx=log_int(10, 80), ny=log_int(10, 80), nz=log_int(6, 90), steps=rng.randint(100, 500))
    elif kind == "bed":
        c.update(nx=log_int(6, 60), ny=log_int(6, 60), nz=log_int(6, 60), steps=rng.randint(10, 50))
    elif kind == "flow":
        c.update(nx=log_int(8, 48), ny=log_int(8, 48), nz=log_int(6, 40), steps=rng.randint(50, 200))
    elif kind == "beam":
        c.update(nx=rng.randint(8, 30), ny=rng.randint(2, 8), nz=rng.randint(2, 8),
                 steps=rng.randint(100, 500))
    elif kind == "column":
        c.update(nx=rng.randint(2, 8), ny=rng.randint(2, 8), nz=log_int(4, 64), floor=rng.randint(9, 16),
                 steps=rng.randint(50, 200))
    elif kind == "adjoint":
        nx, ny = rng.randint(2, 7), rng.randint(2, 7)
        c.update(nx=nx, ny=ny, nz=log_int(4, 48), floor=rng.randint(8, 14), steps=rng.randint(20, 80),
                 every=rng.randint(7, 30))
    else:
        c.update(nu=rng.randint(12, 80), nv=rng.randint(8, 32), resolution=rng.randint(12, 50))
        del c["precision"]
    return c


# ------------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=None)
def _family(count, seed, nodes, scale=1e-3, n_grid=32):
    return W.superellipsoid_family(count, seed, n_grid=n_grid, n_nodes=nodes,
                                   axes=(0.8 * scale, 1.2 * scale))


def _solver(case):
    s = Solver(0, precision=case["precision"])
    if case["kind"] in ("pour", "batch", "flow"):
        s.set_capacity(8, 24)
    elif case["kind"] == "bed":
        s.set_capacity(12, 64)
    return s


def _compressed(scn, moving, steps, closing=3e-3, dt=1e-6):
    """The scenario's lattice after its layers have closed in on one another
    for `steps` steps (heights shrink by about a quarter, overlaps of some
    1e-5 m), at rest: run by the solver itself."""
    v = np.zeros_like(scn.v)
    z = scn.x[:, 2]
    v[moving, 2] = -(z[moving] - z.min()) / closing
    s = Solver(0)
    s.set_capacity(12, 64)
    W.apply(dataclasses.replace(scn, v=v, dt=dt), s)
    s.step(steps)
    st = s.state()
    s.close()
    return dataclasses.replace(scn, x=st["x"], q=st["q"], v=np.zeros_like(scn.v),
                               w=np.zeros_like(scn.w))


def _sizes(case):
    e = np.linspace(math.log(case["lo"]), math.log(case["hi"]), case["count"])
    return [int(round(math.exp(v))) for v in e]


def _scenario(case, seed):
    """The scenario (or, for a batch, the scenarios) of a case."""
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "roll":
        scn = W.single_particle_on_wall(n_nodes=case["nodes"], seed=seed)
        scn.x[0, 0] = -0.3
        return scn
    if kind == "cluster":
        return W.cluster(case["n"], seed=seed, spacing=2.7, scale=1e-2, speed=1.0, spin=20.0, dt=5e-6,
                         periodic=(True, True), templates=_family(3, 101, 256, 1e-2, 16))
    if kind == "packing":
        return W.packing(case["n"], seed, _family(16, 2025, 1000),
                         kn=rng.uniform(5e3, 2e4), mu=rng.uniform(0.2, 0.8), zeta=rng.uniform(0.1, 0.5))
    if kind == "batch":
        # sizes spread evenly over their logarithm; everything else seeded
        t = _family(16, 2025, 1000)
        return [W.packing(n, int(rng.integers(1 << 30)), t, kn=rng.uniform(5e3, 2e4),
                          mu=rng.uniform(0.2, 0.8), zeta=rng.uniform(0.1, 0.5)) for n in _sizes(case)]
    if kind in ("pour", "bed", "flow"):
        scn = W.pour((case["nx"], case["ny"], case["nz"]), seed=seed, templates=_family(16, 2025, 1000))
        if kind == "flow":
            scn.v = rng.normal(0.0, 0.5, size=scn.v.shape)
            # each layer slid sideways, so that bodies cross the periodic faces
            # at every moment of a run
            L = (scn.domain_max - scn.domain_min)[:2]
            off = rng.uniform(0.0, 1.0, size=(case["nz"], 2)) * L
            off = np.repeat(off, case["nx"] * case["ny"], axis=0)
            scn.x[:, :2] = scn.domain_min[:2] + np.mod(scn.x[:, :2] - scn.domain_min[:2] + off, L)
        if kind == "bed":
            scn = _compressed(scn, np.ones(scn.n, bool), 768)
        return scn
    if kind == "beam":
        return W.bonded_beam((case["nx"], case["ny"], case["nz"]), lattice="fcc", seed=seed,
                             tip_speed=float(rng.uniform(0.5, 2.0)))
    scn = W.column((case["nx"], case["ny"], case["nz"]), seed=seed, floor_side=case["floor"])
    tmpl = _family(8, 5, 800)
    scn = dataclasses.replace(scn, templates=tmpl + tmpl)
    _floor_rest(scn, tmpl)
    return _compressed(scn, _moving(scn), 672)


def _moving(scn):
    return ~np.isin(scn.geo, scn.fixed_templates)


def _floor_rest(scn, tmpl):
    """The fixed floor bodies lowered onto the floor with the shapes in use."""
    for i in np.flatnonzero(~_moving(scn)):
        R = W._rotmat(scn.q[i])
        nodes = tmpl[scn.geo[i] - len(tmpl)].nodes.astype(np.float64)
        scn.x[i, 2] = -float(np.min((nodes @ R.T)[:, 2]))


def _mesh(case, seed):
    """A torus with seeded proportions and a smooth seeded bumpiness, scaled
    into a fixed box (off the grid's multiples), so that every seed's grid has
    the same size."""
    rng = np.random.default_rng(seed)
    v, f = G.torus_mesh(1.0, float(rng.uniform(0.3, 0.45)), case["nu"], case["nv"])
    k = rng.integers(2, 5, size=3)
    a = rng.uniform(0.01, 0.04, size=3)
    ph = rng.uniform(0.0, 2 * math.pi, size=3)
    v = v + a * np.sin(k * v[:, [1, 2, 0]] + ph)
    box = np.array([2.8, 2.7, 0.8])
    shift = np.array([0.37, 0.21, 0.43]) * box[0] / case["resolution"]
    v = (v - v.min(0)) / (v.max(0) - v.min(0)) * box - 0.5 * box + shift
    return np.ascontiguousarray(v), f


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mesh":
        return dict(case=case, mesh=G.MeshParticle(*_mesh(case, seed)))
    scn = _scenario(case, seed)
    s = _solver(case)
    if kind == "batch":
        W.apply_batch(scn, s)
        return dict(case=case, solver=s)
    W.apply(scn, s)
    st = dict(case=case, solver=s)
    if kind == "beam":
        st["bonds"] = len(scn.bonds)
    if kind == "adjoint":
        inv = np.array([s.geometry(g)["inv_mass"] for g in range(len(scn.templates))])[scn.geo]
        st["mass"] = np.where(inv > 0.0, 1.0 / np.where(inv > 0.0, inv, 1.0), 0.0)
        st["adjoint"] = Adjoint(s, contacts_per_particle=32)
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "mesh":
        return state["mesh"].build_grid_by_resolution(case["resolution"])[3]
    s = state["solver"]
    if kind == "adjoint":
        # gradients of the final kinetic energy
        adj = state["adjoint"]
        adj.forward(case["steps"], case["every"])
        st = s.state()
        g = adj.backward(v_bar=state["mass"][:, None] * st["v"])
        return dict(state=st, gradient=g)
    s.step(case["steps"])
    out = s.state()
    if kind == "beam":
        out["bonds"] = s.bonds(state["bonds"])
    return out


# --------------------------------------------------------------------- work
def _bodies(case):
    kind = case["kind"]
    if kind == "roll":
        return 1
    if kind in ("cluster", "packing"):
        return case["n"]
    if kind == "batch":
        return sum(_sizes(case))
    if kind == "beam":
        return 4 * case["nx"] * case["ny"] * case["nz"]
    n = case["nx"] * case["ny"] * case["nz"]
    return n + case["floor"] ** 2 if kind in ("column", "adjoint") else n


def work(case):
    """Bytes: per body and step the state read and written once (positions,
    orientation, velocity, spin, force and torque: 88 B in the FP32 build and
    152 B in the FP64 build) and the template and material ids read; per bond
    its 148 B of constants and results; per output value 8 B. Flops: the
    integration of a body (about 200), a bond (about 400), and for bodies in
    contact the transform and sampling of the surface nodes near the partner
    (about 64 nodes of 60 each per touching pair)."""
    kind = case["kind"]
    if kind == "mesh":
        # a torus of unit major radius: extents about 2.8 x 2.8 x 0.8
        nodes = (case["resolution"] + 5) ** 2 * (0.3 * case["resolution"] + 5)
        tris = 2 * case["nu"] * case["nv"]
        return dict(bytes=72.0 * tris + 8.0 * nodes, flops=100.0 * nodes * tris)
    n = _bodies(case)
    state = 88.0 if case["precision"] == "fp32" else 152.0
    per_body = {"roll": 1.0, "cluster": 1.0, "packing": 0.1, "batch": 0.1, "pour": 0.01, "bed": 1.0,
                "flow": 0.3, "beam": 0.0, "column": 1.0, "adjoint": 1.0}[kind]
    bonds = 5.5 * n if kind == "beam" else 0.0
    steps = case["steps"] * (3 if kind == "adjoint" else 1)  # forward, recomputed, reverse
    return dict(bytes=steps * ((2.0 * state + 8.0) * n + 148.0 * bonds) + 152.0 * n,
                flops=steps * (200.0 * n + 400.0 * bonds + 64.0 * 60.0 * per_body * n))


def tolerance(case):
    """A correct implementation at the same precision rounds the stored state
    (FP32: 6e-8 a value, so 6e-10 m on a node of a centimetre body) at every
    step, and a contact force is a stiffness times an overlap of some 1e-6 m:
    the forces of the FP32 build differ from the 64-bit computation below by
    up to 2.7e-3 (a body on a wall), positions by 1e-8; the FP64 build's by
    2.6e-10. The mesh's distances differ by 2.5e-16."""
    if case["kind"] == "mesh":
        return dict(rel=1e-14, max=1e-12)
    if case["precision"] == "fp64":
        return dict(rel=1e-9, max=1e-6)
    return dict(rel=1e-2, max=0.5, differ=1e-3)


# -------------------------------------------------------------------- exact
def exact(case, seed):
    """run()'s answer in 64 bits by plain torch; None where all pairs and all
    nodes would take too long."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    kind = case["kind"]
    if kind == "mesh":
        return _exact_mesh(case, seed, dev)
    limit = {"adjoint": 700, "column": 2500, "beam": 2500}.get(kind, 2500)
    if kind in ("batch", "pour") or _bodies(case) > limit:
        return None
    scn = _scenario(case, seed)
    sim = _Exact(scn, dev)
    if kind != "adjoint":
        with torch.no_grad():
            for _ in range(case["steps"]):
                sim.step()
        return sim.outputs(kind == "beam")
    leaves = [sim.x, sim.q, sim.v, sim.w, sim.kn, sim.ks, sim.mu, sim.zeta, sim.wmu, sim.wzeta]
    for t in leaves:
        t.requires_grad_(True)
    for _ in range(case["steps"]):
        sim.step()
    J = 0.5 * (sim.mass()[:, None] * sim.v.square()).sum()
    g = torch.autograd.grad(J, leaves, allow_unused=True)
    names = ("x", "q", "v", "w", "kn", "ks", "mu", "zeta", "wall_mu", "wall_zeta")
    grad = {k: (torch.zeros_like(t) if d is None else d).detach().cpu().numpy()
            for k, t, d in zip(names, leaves, g)}
    return dict(state=sim.outputs(False), gradient=grad)


def _dot(a, b):
    return (a * b).sum(-1)


def _norm(a):
    """Length with a zero (not undefined) derivative at zero."""
    s = _dot(a, a)
    z = s == 0
    return torch.where(z, torch.zeros_like(s), torch.sqrt(torch.where(z, torch.ones_like(s), s)))


def _unit(a):
    n = _norm(a)
    return a / torch.where(n == 0, torch.ones_like(n), n)[..., None]


def _cross(a, b):
    return torch.linalg.cross(a, b)


def _rot(q, v):
    u = q[..., 1:]
    t = 2.0 * _cross(u.expand_as(v), v)
    return v + q[..., :1] * t + _cross(u.expand_as(v), t)


def _rot_t(q, v):
    return _rot(torch.cat([q[..., :1], -q[..., 1:]], -1), v)


def _matrix(q):
    e = torch.eye(3, dtype=q.dtype, device=q.device)
    return torch.stack([_rot(q, e[k].expand(q.shape[0], 3)) for k in range(3)], -1)


def _sqrt32(x):
    # the contact model takes the roots of its damping in single precision:
    # the value is rounded so, the derivative is the root's
    on = x > 0
    r = torch.where(on, torch.sqrt(torch.where(on, x, torch.ones_like(x))), torch.zeros_like(x))
    return r + (torch.sqrt(x.detach().float()).double() - r.detach())


def _heaviside(phi, eps):
    x = np.clip(-phi / eps, -1.0, 1.0)
    return 0.5 * (1.0 + x + np.sin(math.pi * x) / math.pi)


class _Exact:
    """The timestep of the level-set model for one system, all pairs tested
    node by node: half kick, drift, contacts of every surface node with the
    particles of higher index, the plane walls and the periodic images, bonds,
    half kick."""

    def __init__(self, scn, dev):
        t = functools.partial(torch.tensor, dtype=torch.float64, device=dev)
        self.scn, self.dev, self.dt = scn, dev, scn.dt
        self.x, self.v, self.w, self.q = t(scn.x), t(scn.v), t(scn.w), t(scn.q)
        self.F, self.T = torch.zeros_like(self.x), torch.zeros_like(self.x)
        self.geo = torch.tensor(scn.geo, device=dev, dtype=torch.long)
        self.mat = torch.tensor(scn.mat, device=dev, dtype=torch.long)
        self.g = t(scn.gravity)
        dens = scn.density if isinstance(scn.density, (list, tuple)) else [scn.density] * len(scn.templates)
        self.tmpl = [self._template(tp, 0.0 if k in scn.fixed_templates else dens[k])
                     for k, tp in enumerate(scn.templates)]
        self.walls = [self._template(scn.wall_templates[w[5]], 0.0) for w in scn.walls]
        self.wx = [t(w[0]) for w in scn.walls]
        self.wq = [t(w[3]) for w in scn.walls]
        self.inv_m = t([tp["inv_m"] for tp in self.tmpl])[self.geo]
        self.I = t(np.array([tp["I"] for tp in self.tmpl]))[self.geo]
        self.Iinv = t(np.array([tp["Iinv"] for tp in self.tmpl]))[self.geo]
        self.R = t([tp["radius"] for tp in self.tmpl])[self.geo]
        self.reach = t([tp["reach"] for tp in self.tmpl])[self.geo]
        M = max(len(tp["nodes"]) for tp in self.tmpl)
        nodes = np.full((len(self.tmpl), M, 3), np.nan)
        for k, tp in enumerate(self.tmpl):
            nodes[k, : len(tp["nodes"])] = tp["nodes"]
        self.nodes, self.M = t(nodes), M
        every = self.tmpl + self.walls
        self.origin = t(np.array([tp["origin"] for tp in every]))
        self.h = t([tp["h"] for tp in every])
        self.size = torch.tensor(np.array([tp["size"] for tp in every]), device=dev, dtype=torch.long)
        start = np.cumsum([0] + [tp["sdf"].size for tp in every])[:-1]
        self.start = torch.tensor(start, device=dev, dtype=torch.long)
        self.sdf = t(np.concatenate([tp["sdf"] for tp in every]))

        def zeta(e):
            if scn.damping_ratio:
                return e
            l = math.log(e)
            return -l / float(np.sqrt(np.float32(l * l + math.pi ** 2)))

        m = np.array(scn.materials, dtype=np.float64).reshape(-1, 4)
        self.kn, self.ks, self.mu = t(m[:, 0]), t(m[:, 1]), t(m[:, 2])
        self.zeta = t([zeta(e) for e in m[:, 3]])
        wm = np.array(scn.wall_materials, dtype=np.float64).reshape(-1, 2)
        self.wmu, self.wzeta = t(wm[:, 0]), t([zeta(e) for e in wm[:, 1]])
        self.lo, self.hi = t(scn.domain_min), t(scn.domain_max)
        L = np.asarray(scn.domain_max) - np.asarray(scn.domain_min)
        cs = scn.cell_size if scn.cell_size > 0 else 2.0 * float(self.R.max())
        cells = np.array([int(l / cs) if l > 2.0 * cs else 2 for l in L])
        self.inv_cell = t(cells / L)
        self.history = {}
        self._bonds(scn, t)

    def _template(self, tp, density):
        phi = tp.sdf.astype(np.float64).reshape(tp.size[::-1])  # (z, y, x)
        h, o = tp.spacing, np.asarray(tp.origin, np.float64)
        nodes = tp.nodes.astype(np.float64)
        out = dict(sdf=phi.reshape(-1), h=h, size=np.array(tp.size), inv_m=0.0, I=np.zeros((3, 3)),
                   Iinv=np.zeros((3, 3)))
        if density > 0.0:
            H = _heaviside(phi / h, 1.5)
            p = [o[a] + h * np.arange(tp.size[a]) for a in range(3)]
            P = np.stack(np.meshgrid(*p, indexing="ij"), -1).transpose(2, 1, 0, 3)
            mg = density * h ** 3
            m = mg * H.sum()
            c = mg / m * (H[..., None] * P).sum((0, 1, 2))
            r = P - c
            r2 = (r * r).sum(-1)
            I = mg * (np.eye(3) * (H * r2).sum() - np.einsum("zyx,zyxi,zyxj->ij", H, r, r))
            o, nodes = o - c, nodes - c
            out.update(inv_m=1.0 / m, I=I)
            # the model does not rotate a body whose inertia determinant is
            # below 1e-30 (SI units)
            if abs(np.linalg.det(I)) >= 1e-30:
                out["Iinv"] = np.linalg.inv(I)
        corners = np.array([[o[a] + h * (tp.size[a] - 1) * b[a] for a in range(3)]
                            for b in np.ndindex(2, 2, 2)])
        out.update(origin=o, nodes=nodes, radius=float(np.linalg.norm(nodes, axis=1).max()),
                   reach=float(np.linalg.norm(corners, axis=1).max()))
        return out

    def _bonds(self, scn, t):
        self.nb = len(scn.bonds)
        if not self.nb:
            return
        a = np.array([b[:2] for b in scn.bonds])
        self.bi, self.bj = (torch.tensor(a[:, k], device=self.dev, dtype=torch.long) for k in (0, 1))
        point, normal = t(np.array([b[2] for b in scn.bonds])), t(np.array([b[3] for b in scn.bonds]))
        Rb, L, E, nu, self.st, self.coh, self.mub = t(np.array([b[4:] for b in scn.bonds])).T
        A = math.pi * Rb ** 2
        I = A * Rb ** 2 / 4.0
        self.bR, self.L0 = Rb, L
        self.B1 = E * A / L
        self.B2 = 12.0 * E * I / L
        self.B4 = E / (2.0 * (1.0 + nu)) * 2.0 * I / L
        self.B3 = E * I / L - self.B2 / 4.0 - self.B4 / 2.0
        n = _unit(normal)
        N1 = -n
        ref = torch.where((N1[:, :1].abs() < 0.9), t([1.0, 0.0, 0.0]), t([0.0, 1.0, 0.0]))
        N2 = _unit(_cross(ref, N1))
        N3 = _unit(_cross(N1, N2))
        qi, qj = self.q[self.bi], self.q[self.bj]
        self.li = [_rot_t(qi, d) for d in (N1, N2, N3)]
        self.lj = [_rot_t(qj, d) for d in (-N1, N2, N3)]
        self.pi = _rot_t(qi, point + 0.5 * L[:, None] * n - self.x[self.bi])
        self.pj = _rot_t(qj, point - 0.5 * L[:, None] * n - self.x[self.bj])
        self.active = torch.ones(self.nb, dtype=torch.bool, device=self.dev)
        self.broke = torch.full((self.nb,), -1, dtype=torch.long, device=self.dev)
        self.sigma, self.tau = torch.zeros_like(L), torch.zeros_like(L)
        self.count = 0

    def mass(self):
        return torch.where(self.inv_m > 0, 1.0 / torch.where(self.inv_m > 0, self.inv_m, 1.0), 0.0)

    def kick(self, h):
        free = (self.inv_m > 0)[:, None]
        v = self.v + (self.F * self.inv_m[:, None] + self.g) * h
        Rm = _matrix(self.q)
        Iw = (Rm @ self.I @ Rm.mT @ self.w[..., None])[..., 0]
        Ii = Rm @ self.Iinv @ Rm.mT
        w = self.w + (Ii @ (self.T - _cross(self.w, Iw))[..., None])[..., 0] * h
        self.v, self.w = torch.where(free, v, self.v), torch.where(free, w, self.w)

    def drift(self):
        self.x = self.x + self.v * self.dt
        q, d = self.q, self.w * (0.5 * self.dt)
        s = -_dot(q[:, 1:], d)
        u = q[:, :1] * d + _cross(d, q[:, 1:])
        self.q = _unit(q + torch.cat([s[:, None], u], -1))

    def sample(self, local, tid):
        """Inside flag, level-set value and gradient (taken at the cell's
        lower x face for its y and z parts) of points in template frames."""
        with torch.no_grad():
            cell = torch.floor((local - self.origin[tid]) / self.h[tid][..., None])
            sz = self.size[tid]
            inside = ((cell >= 0) & (cell < sz - 1)).all(-1)
            c = torch.where(inside[..., None], cell, torch.zeros_like(cell)).long()
            base = self.start[tid] + c[..., 0] + sz[..., 0] * (c[..., 1] + sz[..., 1] * c[..., 2])
            ny, nz = sz[..., 0], sz[..., 0] * sz[..., 1]
            f = {(i, j, k): self.sdf[base + i + ny * j + nz * k] for k in (0, 1) for j in (0, 1) for i in (0, 1)}
        r = (local - self.origin[tid]) / self.h[tid][..., None] - c
        x, y, z = r.unbind(-1)

        def lerp(a, b, s):
            return a * (1 - s) + b * s

        fx = {(j, k): lerp(f[0, j, k], f[1, j, k], x) for j in (0, 1) for k in (0, 1)}
        val = lerp(lerp(fx[0, 0], fx[1, 0], y), lerp(fx[0, 1], fx[1, 1], y), z)
        dx = {(j, k): f[1, j, k] - f[0, j, k] for j in (0, 1) for k in (0, 1)}
        gx = lerp(lerp(dx[0, 0], dx[1, 0], y), lerp(dx[0, 1], dx[1, 1], y), z)
        gy = lerp(f[0, 1, 0] - f[0, 0, 0], f[0, 1, 1] - f[0, 0, 1], z)
        gz = lerp(f[0, 0, 1] - f[0, 0, 0], f[0, 1, 1] - f[0, 1, 0], y)
        return inside, val, torch.stack([gx, gy, gz], -1)

    def contacts(self, A, xT, qT, tid, sphere, rT):
        """Contacts of the candidate pairs (A, target): pair and node ids."""
        got = []
        with torch.no_grad():
            for s in range(0, len(A), 4096):
                a = A[s:s + 4096]
                p = _rot(self.q[a][:, None], self.nodes[self.geo[a]]) + self.x[a][:, None]
                rel = p - xT[s:s + 4096][:, None]
                ok = ~torch.isnan(p[..., 0])
                if sphere:
                    ok &= _dot(rel, rel) <= (rT[s:s + 4096] ** 2)[:, None]
                k = ok.nonzero()
                local = _rot_t(qT[s + k[:, 0]], rel[k[:, 0], k[:, 1]])
                inside, val, _ = self.sample(local, tid[s + k[:, 0]])
                k = k[inside & (-val >= 0)]
                got.append(torch.stack([k[:, 0] + s, k[:, 1]], 1))
        return torch.cat(got) if got else torch.zeros((0, 2), dtype=torch.long, device=self.dev)

    def geometry(self, pair, node, A, xT, qT, tid, xA):
        a = A[pair]
        p = _rot(self.q[a], self.nodes[self.geo[a], node]) + xA[a]
        _, val, grad = self.sample(_rot_t(qT[pair], p - xT[pair]), tid[pair])
        n = _unit(_rot(qT[pair], grad))
        return p + n * (-0.5 * val)[:, None], n, -val

    def law(self, name, key, pc, n, ov, vc, kn, ks, mu, zeta, eff):
        """Spring-dashpot with Coulomb cap; the spring of a node and target is
        carried from the step before."""
        old_key, old = self.history.get(name, (None, None))
        prev = torch.zeros_like(pc)
        if old_key is not None and len(old_key) and len(key):
            at = torch.searchsorted(old_key, key).clamp(max=len(old_key) - 1)
            prev = torch.where((old_key[at] == key)[:, None], old[at], prev)
        cn, ct = 2.0 * zeta * _sqrt32(eff * kn), 2.0 * zeta * _sqrt32(eff * ks)
        vn = n * _dot(vc, n)[:, None]
        Fn = n * (kn * ov)[:, None] - vn * cn[:, None]
        vt = vc - vn
        p1 = prev - n * _dot(prev, n)[:, None]
        a1 = _norm(p1)
        p1 = p1 * torch.where(a1 > 1e-20, _norm(prev) / torch.where(a1 > 1e-20, a1, 1.0), 1.0)[:, None]
        s = p1 + vt * self.dt
        Fs = -s * ks[:, None] - vt * ct[:, None]
        af, cap = _norm(Fs), mu * _norm(Fn)
        slip = (af > 1e-20) & (af > cap)
        Fc = Fs * (cap / torch.where(slip, af, 1.0))[:, None]
        s = torch.where(slip[:, None], -(Fc + vt * ct[:, None]) / ks[:, None], s)
        s = torch.where(((mu > 0) & (ks > 0))[:, None], s, torch.zeros_like(s))
        on = (ov > 0)[:, None]
        s = torch.where(on, s, torch.zeros_like(s))
        F = torch.where(on, Fn - s * ks[:, None] - vt * ct[:, None], torch.zeros_like(Fn))
        order = torch.argsort(key)
        self.history[name] = (key[order], s[order])
        return F

    def pair_law(self, name, A, B, pair, node, pc, n, ov, xA, xB):
        a, b = A[pair], B[pair]
        ma, mb = self.mat[a], self.mat[b]
        kn = self.kn[ma] * self.kn[mb] / (self.kn[ma] + self.kn[mb])
        ks = self.ks[ma] * self.ks[mb] / (self.ks[ma] + self.ks[mb])
        im = self.inv_m[a] + self.inv_m[b]
        eff = torch.where(im > 0, 1.0 / torch.where(im > 0, im, 1.0), 0.0)
        mu, zeta = torch.minimum(self.mu[ma], self.mu[mb]), torch.maximum(self.zeta[ma], self.zeta[mb])
        ra, rb = pc - xA[a], pc - xB[pair]
        vc = self.v[a] + _cross(self.w[a], ra) - self.v[b] - _cross(self.w[b], rb)
        N = len(self.x)
        F = self.law(name, (a * N + b) * self.M + node, pc, n, ov, vc, kn, ks, mu, zeta, eff)
        own = a == b  # a body and its own image: the image takes no force
        self.add(a, F, _cross(ra, F))
        self.add(b, torch.where(own[:, None], 0.0, -F), torch.where(own[:, None], 0.0, _cross(rb, -F)))

    def add(self, i, F, T):
        self.F = self.F.index_add(0, i, F)
        self.T = self.T.index_add(0, i, T)

    def step(self):
        h = 0.5 * self.dt
        self.kick(h)
        self.drift()
        N = len(self.x)
        x, scn = self.x, self.scn
        valid = ((x >= self.lo) & (x < self.hi)).all(-1)
        # particle pairs and walls are found before the periodic wrap
        d = torch.cdist(x.detach(), x.detach(), compute_mode="donot_use_mm_for_euclid_dist")
        near = (d <= 1.001 * (self.R[:, None] + self.R[None])) & valid[None]
        A, B = torch.triu(near, 1).nonzero().T
        found = self.contacts(A, x[B], self.q[B], self.geo[B], True, self.R[B])
        pp = (A, B, found[:, 0], found[:, 1],
              self.geometry(found[:, 0], found[:, 1], A, x[B], self.q[B], self.geo[B], x))
        pw = []
        for k, (wx, wq) in enumerate(zip(self.wx, self.wq)):
            tid = len(self.tmpl) + k
            inside, val, _ = self.sample(_rot_t(wq, x.detach() - wx),
                                         torch.full((N,), tid, device=self.dev, dtype=torch.long))
            A = ((val <= 1.01 * self.R) | ~inside).nonzero()[:, 0]  # plane walls: unit slope
            X, Q, Ti = wx.expand(len(A), 3), wq.expand(len(A), 4), torch.full_like(A, tid)
            found = self.contacts(A, X, Q, Ti, False, None)
            pw.append((k, A, found[:, 0], found[:, 1],
                       self.geometry(found[:, 0], found[:, 1], A, X, Q, Ti, x)))
        images = []
        L = self.hi - self.lo
        for axis in (0, 1):
            if scn.periodic[axis]:
                c = self.x[:, axis]
                shift = torch.where(c < self.lo[axis], L[axis], torch.where(c >= self.hi[axis], -L[axis], 0.0))
                e = torch.zeros(3, device=self.dev, dtype=torch.float64)
                e[axis] = 1.0
                self.x = self.x + shift[:, None] * e
                images.append(((axis,), self.x))
        if all(scn.periodic):
            images.append(((0, 1), self.x))
        ghosts = []
        for axes, xg in images:
            cell = ((xg - self.lo) * self.inv_cell).detach()
            first = torch.ones(N, dtype=torch.bool, device=self.dev)
            off = torch.zeros(3, device=self.dev, dtype=torch.float64)
            for a in axes:
                first &= cell[:, a].trunc() == 0
                off[a] = L[a]
            pos = xg + torch.where(first[:, None], off, torch.zeros_like(off))
            out = ((pos < self.lo) | (pos >= self.hi)).any(-1)
            xa = self.x.detach()
            d = torch.cdist(xa, pos.detach(), compute_mode="donot_use_mm_for_euclid_dist")
            A, B = ((d <= 1.001 * (self.R[:, None] + self.reach[None])) & out[None]).nonzero().T
            found = self.contacts(A, pos[B], self.q[B], self.geo[B], False, None)
            ghosts.append((axes, A, B, found[:, 0], found[:, 1], pos,
                           self.geometry(found[:, 0], found[:, 1], A, pos[B], self.q[B], self.geo[B], self.x)))
        self.F, self.T = torch.zeros_like(self.F), torch.zeros_like(self.T)
        A, B, pair, node, (pc, n, ov) = pp
        self.pair_law("pp", A, B, pair, node, pc, n, ov, self.x, self.x[B])
        for k, A, pair, node, (pc, n, ov) in pw:
            a = A[pair]
            ma, mw = self.mat[a], scn.walls[k][4]
            im = self.inv_m[a]
            eff = torch.where(im > 0, 1.0 / torch.where(im > 0, im, 1.0), 0.0)
            r = pc - self.x[a]
            vc = self.v[a] + _cross(self.w[a], r)
            F = self.law(("pw", k), a * self.M + node, pc, n, ov, vc, self.kn[ma], self.ks[ma],
                         torch.where(self.mu[ma] <= self.wmu[mw], self.mu[ma], self.wmu[mw]),
                         torch.where(self.zeta[ma] >= self.wzeta[mw], self.zeta[ma], self.wzeta[mw]), eff)
            self.add(a, F, _cross(r, F))
        for axes, A, B, pair, node, pos, (pc, n, ov) in ghosts:
            self.pair_law(axes, A, B, pair, node, pc, n, ov, self.x, pos[B])
        if self.nb:
            self.bond_forces()
        self.kick(h)

    def bond_forces(self):
        i, j = self.bi, self.bj
        qi, qj = self.q[i], self.q[j]
        n1i, n2i, n3i = (_rot(qi, d) for d in self.li)
        n1j, n2j, n3j = (_rot(qj, d) for d in self.lj)
        ri, rj = _rot(qi, self.pi), _rot(qj, self.pj)
        rij = self.x[i] + ri - self.x[j] - rj
        D = _norm(rij)
        nij = _unit(rij)
        e = -nij
        dn = n1j - n1i
        F = e * (self.B1 * (D - self.L0))[:, None] \
            + (dn - e * _dot(dn, e)[:, None]) * (self.B2 / (2.0 * D))[:, None]
        tb = _cross(n1j, n1i) * self.B3[:, None] - (_cross(n2j, n2i) + _cross(n3j, n3i)) * (0.5 * self.B4)[:, None]
        Mi = _cross(e, n1i) * (-0.5 * self.B2)[:, None] + tb
        Mj = _cross(e, n1j) * (0.5 * self.B2)[:, None] - tb
        Fn = _dot(F, nij)
        Tt = _dot(tb, nij)
        A = math.pi * self.bR ** 2
        I = A * self.bR ** 2 / 4.0
        sigma = -Fn / A + _norm(tb - nij * Tt[:, None]) / I * self.bR
        tau = _norm(F - nij * Fn[:, None]) / A + Tt.abs() / (2.0 * I) * self.bR
        on = self.active
        zero = torch.zeros_like(F)
        F, Mi, Mj = (torch.where(on[:, None], t, zero) for t in (F, Mi, Mj))
        self.add(i, F, Mi + _cross(ri, F))
        self.add(j, -F, Mj + _cross(rj, -F))
        self.sigma, self.tau = torch.where(on, sigma, 0.0), torch.where(on, tau, 0.0)
        fails = on & (((self.st > 0) & (sigma > self.st)) | ((self.coh > 0) & (tau > self.coh - self.mub * sigma)))
        self.broke = torch.where(fails, torch.full_like(self.broke, self.count), self.broke)
        self.active = on & ~fails
        self.count += 1

    def outputs(self, bonds):
        out = {k: getattr(self, k).detach().cpu().numpy() for k in ("x", "v", "w", "q", "F", "T")}
        if bonds:
            out["bonds"] = dict(active=self.active.int().cpu().numpy(),
                                break_step=self.broke.int().cpu().numpy(),
                                sigma=self.sigma.cpu().numpy(), tau=self.tau.cpu().numpy())
        return out


def _exact_mesh(case, seed, dev):
    """Signed distances of the grid nodes: the least distance to a triangle
    (its inner region or an edge), negative where the triangles' solid angles
    add up to a full sphere."""
    v, f = _mesh(case, seed)
    # nodes at multiples of the spacing covering the mesh's box and two layers
    h = (v.max(0) - v.min(0)).max() / case["resolution"]
    lo = h * np.floor((v.min(0) - 2.0 * h) / h)
    hi = h * np.ceil((v.max(0) + 2.0 * h) / h)
    size = np.floor((hi - lo) / h + 0.5).astype(int) + 1
    ax = [lo[a] + h * np.arange(size[a]) for a in range(3)]
    z, y, x = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    pts = torch.tensor(np.stack([x, y, z], -1).reshape(-1, 3), device=dev)
    a, b, c = (torch.tensor(v[f[:, k]], device=dev)[None] for k in range(3))
    n = _cross(b - a, c - a)
    nn = _dot(n, n)

    def segment(p, s, e):
        d = e - s
        t = (_dot(p - s, d) / _dot(d, d)).clamp(0.0, 1.0)[..., None]
        r = p - s - d * t
        return _dot(r, r)

    out = []
    for k in range(0, len(pts), max(1, (1 << 24) // len(f))):
        p = pts[k:k + max(1, (1 << 24) // len(f))][:, None]
        pa, pb, pc = a - p, b - p, c - p
        d2 = torch.minimum(torch.minimum(segment(p, a, b), segment(p, b, c)), segment(p, c, a))
        inner = ((_dot(_cross(b - a, -pa), n) >= 0) & (_dot(_cross(c - b, -pb), n) >= 0)
                 & (_dot(_cross(a - c, -pc), n) >= 0))
        d2 = torch.where(inner, torch.minimum(d2, _dot(pa, n.expand_as(pa)) ** 2 / nn), d2).amin(1)
        la, lb, lc = _norm(pa), _norm(pb), _norm(pc)
        den = la * lb * lc + _dot(pa, pb) * lc + _dot(pb, pc) * la + _dot(pc, pa) * lb
        solid = 2.0 * torch.atan2(_dot(pa, _cross(pb, pc)), den)
        inside = (solid.sum(1) / (4.0 * math.pi)).abs() > 0.5
        out.append(torch.where(inside, -d2.sqrt(), d2.sqrt()))
    return torch.cat(out).cpu().numpy()
