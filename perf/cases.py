"""What a user of this framework has it compute, at the sizes it is used at.

A case is a dict of plain values; its "kind" is one of

  collision  the two colliding discs of the reference's test program, advanced
             one velocity-Verlet step operator by operator, energy read after it
  steps      a dam break in a tank (2D or 3D) advanced some fused steps by one
             step() call, then its positions, velocities and densities read back
  operators  the dam break advanced through the collapse_dry program's own
             operators, call by call, then read back
  vortices   a batch of periodic Taylor-Green boxes of uneven size, advanced by
             one Batch.step() call, every box read back
  tanks      a batch of small 2D dam breaks of uneven size (the small requests
             of a served stream), advanced a short quantum, every tank read back
  probes     SmoothedParticles.sum at scattered points of a 3D tank

Fluid particles lie on a lattice disturbed by a tenth of the spacing and move
with a divergence-free field of a few m/s, as they do in the middle of a run;
the walls keep their lattice.  The mixed mode forms its pair sums in FP32, so
the densities and velocities of mixed cases are taken as FP32, as a viewer
takes them; positions, and every output of the FP64 mode, are FP64.

exact() restates the same physics in plain torch, in FP64, from the inputs.
"""
import math
import pathlib
import random
import sys

import numpy as np
import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parents[1] / "smoothedparticles.jl_amd"))

import smoothedparticles_hip as sp  # noqa: E402

RHO0 = 1000.0
GRAVITY = 9.8
SPEED = 2.0  # m/s, amplitude of the tanks' initial flow
# A step's arithmetic per accepted ordered pair: 15 operations for the
# density (or continuity) sum, 45 for the force.
FLOPS_PER_PAIR = 60
# Neighbours within R = 4.8 dr on a square / cubic lattice, without the own one.
NEIGHBOURS = {2: 68, 3: 460}
# exact() enumerates the candidates of the 9 or 27 cells; above this many over
# all passes it would take too long.
EXACT_CANDIDATES = 4.0e10


# ---------------------------------------------------------------- cases --
def listed():
    return [
        # the reference's own test program: 2.5k particles, ten synchronous
        # calls per time step -- latency of single small calls
        dict(name="collision_2d_operators", kind="collision", dr=0.02),
        # the reference's dam break in two dimensions, 6514 particles, plain
        # FP64: the CPU-sized simulation a user starts with
        dict(name="dam2d_small_fp64", kind="steps", dim=2, dr=0.02, precision="fp64",
             scheme="wcsph_se_rho0", steps=50),
        # a 2D tank of a design study: about 100k particles, mixed
        dict(name="dam2d_100k_mixed", kind="steps", dim=2, dr=0.0047, precision="mixed",
             scheme="wcsph_se_rho0", steps=40),
        # a small 3D tank (100k particles), where tiles hardly fill the chip
        dict(name="dam3d_100k_mixed", kind="steps", dim=3, dr=0.04, precision="mixed",
             scheme="wcsph_se_rho0", steps=16),
        # the headline: 5.75M particles in 3D, mixed, between two frames
        dict(name="dam3d_5M_mixed", kind="steps", dim=3, dr=0.0079, precision="mixed",
             scheme="wcsph_se_rho0", steps=10),
        # the FP64 drop-in on 1.7M particles in 3D
        dict(name="dam3d_2M_fp64", kind="steps", dim=3, dr=0.0125, precision="fp64",
             scheme="wcsph_se_rho0", steps=4),
        # the reference's dry collapse as one fused scheme (two cell lists a
        # step, laminar viscosity, density diffusion), 0.5M particles in 3D
        dict(name="collapse3d_500k_mixed", kind="steps", dim=3, dr=0.02, precision="mixed",
             scheme="collapse_dry", steps=5),
        # the reference's dry collapse driven call by call, as a program ported
        # line by line does it: FP64, 2D, about 25k particles
        dict(name="collapse2d_operators_fp64", kind="operators", dim=2, dr=0.0097,
             precision="fp64", iterations=5),
        # 256 periodic vortices of 2k to 60k particles (5M in all) in one batch
        dict(name="vortices_256_mixed", kind="vortices", boxes=256, lo=2000, hi=60000,
             precision="mixed", steps=16),
        # a few periodic vortices in FP64, the run that others are checked by
        dict(name="vortices_16_fp64", kind="vortices", boxes=16, lo=2000, hi=60000,
             precision="fp64", steps=20),
        # small served requests: 24 tanks of 1k to 8k particles, a short quantum
        dict(name="tanks_24_mixed", kind="tanks", boxes=24, lo=1000, hi=8000,
             precision="mixed", steps=10),
        # a frame's worth of interpolation points in a 0.5M-particle tank
        dict(name="probes_65k", kind="probes", dim=3, dr=0.02, probes=65536),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["collision", "steps", "steps", "steps", "steps", "operators", "vortices",
                       "tanks", "probes"])
    if kind == "collision":
        return dict(kind=kind, dr=round(_log(rng, 0.008, 0.04), 5))
    if kind == "steps":
        dim = rng.choice([2, 3])
        scheme = rng.choice(["wcsph_se_rho0", "wcsph_se_rho0", "collapse_dry"])
        precision = rng.choice(["mixed", "fp64"])
        if dim == 2:
            dr = _log(rng, 0.0025, 0.05)
        else:  # an FP64 or two-list step costs more: the largest tanks are mixed
            dr = _log(rng, 0.009 if precision == "mixed" and scheme != "collapse_dry" else 0.0135,
                      0.08)
        steps = rng.randint(5, 12) if dim == 2 else rng.randint(3, 8)
        return dict(kind=kind, dim=dim, dr=round(dr, 6), precision=precision, scheme=scheme,
                    steps=steps)
    if kind == "operators":
        return dict(kind=kind, dim=2, dr=round(_log(rng, 0.006, 0.04), 5),
                    precision=rng.choice(["fp64", "mixed"]), iterations=rng.randint(2, 6))
    if kind == "vortices":
        lo = int(_log(rng, 1000, 8000))
        return dict(kind=kind, boxes=int(_log(rng, 2, 128)), lo=lo,
                    hi=int(lo * rng.uniform(2.0, 7.0)), precision=rng.choice(["mixed", "fp64"]),
                    steps=rng.randint(5, 10))
    if kind == "tanks":
        lo = int(_log(rng, 1000, 4000))
        return dict(kind=kind, boxes=rng.randint(2, 48), lo=lo, hi=int(lo * rng.uniform(2.0, 8.0)),
                    precision=rng.choice(["mixed", "mixed", "fp64"]), steps=rng.randint(4, 10))
    return dict(kind=kind, dim=3, dr=round(_log(rng, 0.015, 0.05), 5),
                probes=int(_log(rng, 500, 100000)))


# --------------------------------------------------------------- inputs --
def _grid(*axes):
    """The points of a product of index ranges, first axis outermost."""
    g = np.meshgrid(*[np.asarray(a, dtype=np.float64) for a in axes], indexing="ij")
    return np.stack([a.reshape(-1) for a in g], axis=1)


class Inputs:
    """One system's arrays (reference order), box and parameters."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    @property
    def params(self):
        return dict(m=self.m, rho0=self.rho0, c=self.c, alpha=self.alpha, hs=self.hs, mu=self.mu,
                    nu=self.nu, g=tuple(self.g), dt=self.dt)


def _tank(dim, dr, seed, scheme):
    """A block of fluid of 1 x 2 (1 x 1 x 2) m at one end of a 4 m long, 3 m
    high tank without a lid, walls of three layers; vertical axis last."""
    top = 2.0
    ext = (4.0, 3.0) if dim == 2 else (4.0, 1.0, 3.0)
    block = (1.0, top) if dim == 2 else (1.0, 1.0, top)
    count = [int(math.floor(e / dr + 1e-9)) for e in ext]      # last lattice index inside
    rng = np.random.default_rng([seed, dim, int(round(dr * 1e9))])
    fluid = _grid(*[range(int(math.floor(b / dr + 1e-9)) + 1) for b in block]) * dr
    fluid += rng.uniform(-0.1 * dr, 0.1 * dr, fluid.shape)
    fluid = np.abs(fluid)  # the walls' first layer lies at -dr: stay at or above 0
    L = 3
    below, above = range(-L, 0), [range(c + 1, c + 1 + L) for c in count]
    inside = [range(c + 1) for c in count]
    whole = [range(-L, c + 1 + L) for c in count]
    walls = [_grid(*whole[:-1], below)]
    for side in (below, above[0]):
        walls.append(_grid(side, *whole[1:-1], inside[-1]))
    if dim == 3:
        for side in (below, above[1]):
            walls.append(_grid(inside[0], side, inside[-1]))
    walls = np.concatenate(walls) * dr
    n = len(fluid)
    x = np.zeros((n + len(walls), 3))
    x[:n, :dim] = fluid
    x[n:, :dim] = walls
    v = np.zeros_like(x)
    # psi = sin(pi x) sin(pi z / 2): no flow through the block's sides
    amp = SPEED * rng.uniform(0.6, 1.0)
    px, pz = math.pi * fluid[:, 0], 0.5 * math.pi * fluid[:, -1]
    v[:n, 0] = 0.5 * amp * np.sin(px) * np.cos(pz)
    v[:n, dim - 1] = -amp * np.cos(px) * np.sin(pz)
    kind = np.zeros(len(x))
    kind[n:] = 1.0
    g = np.zeros(3)
    g[dim - 1] = -GRAVITY
    c = 50.0
    P = RHO0 * GRAVITY * (top - x[:, dim - 1])
    rho = RHO0 + P / (c * c)
    lo, hi = np.zeros(3), np.zeros(3)
    lo[:dim] = -3.5 * dr
    hi[:dim] = np.array(ext) + 3.5 * dr
    dry = scheme == "collapse_dry"
    return Inputs(dim=dim, x=x, v=v, rho=rho, P=P, type=kind, lo=lo, hi=hi, h=4.8 * dr, box=None,
                  m=RHO0 * dr ** dim, rho0=RHO0, c=c, alpha=0.0 if dry else 0.02, hs=2.4 * dr,
                  mu=8.4e-4 if dry else 0.0, nu=1.0e-6 if dry else 0.0, g=g,
                  dt=0.1 * 2.4 * dr / c)


def _discs(dr, seed):
    """Two discs of radius 0.4 m that meet at 2 m/s."""
    rng = np.random.default_rng([seed, 2, int(round(dr * 1e9))])
    parts, speeds = [], []
    for sign in (-1.0, 1.0):
        k = int(math.ceil(0.6 / dr))
        pts = _grid(range(-2 * k, 2 * k + 1), range(-2 * k, 2 * k + 1)) * dr
        centre = np.array([0.5 * sign, 0.1 * sign])
        pts = pts[((pts - centre) ** 2).sum(axis=1) <= 0.16]
        parts.append(pts)
        speeds.append(np.full(len(pts), -sign))
    pts = np.concatenate(parts)
    x = np.zeros((len(pts), 3))
    x[:, :2] = pts + rng.uniform(-0.05 * dr, 0.05 * dr, pts.shape)
    v = np.zeros_like(x)
    v[:, 0] = np.concatenate(speeds) * rng.uniform(0.9, 1.1)
    h = 2.4 * dr
    zero = np.zeros(len(x))
    return Inputs(dim=2, x=x, v=v, rho=zero, P=zero, type=zero, lo=np.array([-10.0, -10.0, 0.0]),
                  hi=np.array([10.0, 10.0, 0.0]), h=h, box=None, m=RHO0 * dr * dr, rho0=RHO0,
                  c=20.0, alpha=0.0, hs=h, mu=0.0, nu=0.0, g=np.zeros(3), dt=0.1 * h / 20.0)


def _vortex(side, reynolds, seed):
    """A Taylor-Green vortex on side x side particles of the periodic unit box."""
    dr = 1.0 / side
    rng = np.random.default_rng([seed, side])
    x = np.zeros((side * side, 3))
    x[:, :2] = (_grid(range(side), range(side)) + 0.5) * dr
    x[:, :2] += rng.uniform(-0.1 * dr, 0.1 * dr, (side * side, 2))
    v = np.zeros_like(x)
    tp = 2.0 * math.pi
    amp = rng.uniform(0.8, 1.0)
    v[:, 0] = amp * np.sin(tp * x[:, 0]) * np.cos(tp * x[:, 1])
    v[:, 1] = -amp * np.cos(tp * x[:, 0]) * np.sin(tp * x[:, 1])
    one = np.ones(len(x))
    return Inputs(dim=2, x=x, v=v, rho=one, P=0.0 * one, type=0.0 * one, lo=np.zeros(3),
                  hi=np.array([1.0, 1.0, 0.0]), h=4.8 * dr, box=np.array([1.0, 1.0]), m=dr * dr,
                  rho0=1.0, c=10.0, alpha=0.0, hs=2.4 * dr, mu=1.0 / reynolds, nu=0.0,
                  g=np.zeros(3), dt=0.1 * 2.4 * dr / 10.0)


def _sizes(case):
    """The batch's uneven sizes: fixed by the case, log-uniform in [lo, hi]."""
    r = random.Random(f"{case['boxes']} {case['lo']} {case['hi']}")
    return [_log(r, case["lo"], case["hi"]) for _ in range(case["boxes"])]


def _systems(case, seed):
    """The inputs of every system of a case."""
    kind = case["kind"]
    if kind == "collision":
        return [_discs(case["dr"], seed)]
    if kind == "vortices":
        r = random.Random(seed)
        return [_vortex(max(16, round(math.sqrt(n))), r.uniform(50.0, 1000.0), seed + 1000 * k)
                for k, n in enumerate(_sizes(case))]
    if kind == "tanks":
        return [_tank(2, math.sqrt(2.0 / n), seed + 1000 * k, "wcsph_se_rho0")
                for k, n in enumerate(_sizes(case))]
    scheme = {"operators": "collapse_dry"}.get(kind, case.get("scheme", "wcsph_se_rho0"))
    return [_tank(case["dim"], case["dr"], seed, scheme)]


def _probe_points(case, inp, seed):
    """Points of the fluid's box and a little around it."""
    rng = np.random.default_rng([seed, 7])
    lo, hi = np.array([-0.02, -0.02, -0.02]), np.array([1.05, 1.02, 2.05])
    return lo + rng.random((case["probes"], 3)) * (hi - lo)


# ----------------------------------------------------------------- runs --
def prepare(case, seed):
    """The system (or batch) as a program holds it before its time loop:
    particles on the device, reference densities or first forces set."""
    kind = case["kind"]
    systems = _systems(case, seed)
    if kind in ("vortices", "tanks"):
        b = sp.Batch(case["precision"])
        ids = [b.add(s.x, s.h, s.lo, s.hi, periodic=s.box is not None, v=s.v, rho=s.rho, P=s.P,
                     type=s.type, **s.params) for s in systems]
        b.init_rho0()
        return dict(case=case, batch=b, ids=ids)
    s = systems[0]
    precision = "fp64" if kind in ("collision", "probes") else case["precision"]
    g = sp.ParticleSystem(sp.Box(*s.lo, *s.hi), s.h, precision)
    g.add_particles(s.x, v=s.v, rho=s.rho, P=s.P, type=s.type)
    p = s.params
    if kind == "collision":
        sp.create_cell_list(g)
        sp.apply(g, sp.find_rho0, self=True, **p)
        sp.apply(g, sp.find_rho, self=True, **p)
        sp.apply(g, sp.find_pressure_rho0, **p)
        sp.apply(g, sp.internal_force_rho0, **p)
        return dict(case=case, system=g, params=p, ops=sp.program_operators("test_collision_2d"))
    if kind == "probes":
        sp.create_cell_list(g)
        return dict(case=case, system=g, params=p, points=_probe_points(case, s, seed))
    if kind == "operators" or case["scheme"] == "collapse_dry":
        sp.collapse_dry_init(g, **p)
    else:
        sp.init_reference_density(g, **p)
    return dict(case=case, system=g, params=p, ops=sp.program_operators("collapse_dry"))


def _outputs(precision, x, v, rho):
    out = dict(x=torch.from_numpy(x), v=torch.from_numpy(v), rho=torch.from_numpy(rho))
    if precision == "mixed":
        out["v"], out["rho"] = out["v"].float(), out["rho"].float()
    return out


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind in ("vortices", "tanks"):
        b = state["batch"]
        b.step(case["steps"], scheme="wcsph_se_rho0")
        got = {f: np.concatenate([b.get(i, f) for i in state["ids"]]) for f in ("x", "v", "rho")}
        return _outputs(case["precision"], **got)
    g, p = state["system"], state["params"]
    if kind == "probes":
        return sp.probe_sums(g, state["points"], fluid_only=True, **p)
    if kind == "collision":
        ops = state["ops"]
        sp.apply(g, ops["accelerate!"], **p)
        sp.apply(g, ops["move!"], **p)
        sp.create_cell_list(g)
        sp.apply(g, ops["reset_rho!"])
        sp.apply(g, ops["find_rho!"], self=True, **p)
        sp.apply(g, ops["find_pressure!"], **p)
        sp.apply(g, ops["reset_a!"])
        sp.apply(g, ops["internal_force!"], **p)
        sp.apply(g, ops["accelerate!"], **p)
        out = _outputs("fp64", g.get("x"), g.get("v"), g.get("rho"))
        out["energy"] = sp.energy(g, "collision", **p)
        return out
    if kind == "operators":
        ops = state["ops"]
        for _ in range(case["iterations"]):
            sp.apply(g, ops["accelerate!"], **p)
            sp.apply(g, ops["move!"], **p)
            sp.create_cell_list(g)
            sp.apply(g, ops["balance_of_mass!"], **p)
            sp.apply(g, ops["find_pressure!"], **p)
            sp.apply(g, ops["move!"], **p)
            sp.create_cell_list(g)
            sp.apply(g, ops["internal_force!"], **p)
            sp.apply(g, ops["accelerate!"], **p)
    else:
        sp.step(g, case["steps"], scheme=case["scheme"], **p)
    return _outputs(case["precision"], g.get("x"), g.get("v"), g.get("rho"))


# ----------------------------------------------------------------- work --
def _particles(case):
    """Particles of a case (walls counted by their area)."""
    kind = case["kind"]
    if kind == "vortices":
        return sum(max(16, round(math.sqrt(n))) ** 2 for n in _sizes(case))
    if kind == "collision":
        return 2 * math.pi * 0.16 / case["dr"] ** 2

    def tank(dim, dr):
        if dim == 2:
            return 2.0 / dr ** 2 + 3 * (4.0 + 3.0 + 3.0) / dr
        return 2.0 / dr ** 3 + 3 * (4.0 + 2 * 3.0 + 2 * 12.0) / dr ** 2

    if kind == "tanks":
        return sum(tank(2, math.sqrt(2.0 / n)) for n in _sizes(case))
    return tank(case["dim"], case["dr"])


def work(case):
    kind = case["kind"]
    n = _particles(case)
    if kind == "probes":
        near = NEIGHBOURS[3] + 1
        return dict(bytes=case["probes"] * (3 + 4) * 8.0 + n * 7 * 8.0,
                    flops=case["probes"] * near * 25.0)
    dim = case.get("dim", 2)
    near = 18 if kind == "collision" else NEIGHBOURS[dim]  # R = 2.4 dr: 18 on the lattice
    steps = case.get("steps", case.get("iterations", 1))
    # a step reads x, v, rho, rho0 and the type and writes x, v and rho, FP64
    return dict(bytes=steps * n * (9 + 7) * 8.0, flops=steps * n * near * float(FLOPS_PER_PAIR))


# ---------------------------------------------------------------- exact --
def _neighbours(x, h, box):
    """The pairs p != q within h as chunks (p, q, x_p - x_q, r)."""
    n, dim = x.shape
    dev = x.device
    if box is None:
        lo = x.min(dim=0).values
        cell = torch.full((dim,), h, dtype=x.dtype, device=dev)
        c = torch.floor((x - lo) / cell).long()
        count = [int(v) + 1 for v in c.max(dim=0).values]
    else:
        count = [int(math.floor(b / h)) for b in box]
        cell = torch.tensor([b / k for b, k in zip(box, count)], dtype=x.dtype, device=dev)
        c = torch.floor((x - torch.floor(x)) / cell).long()
    lim = torch.tensor(count, device=dev)
    c = torch.minimum(c.clamp(min=0), lim - 1)

    def key_of(cells):
        k = cells[:, 0]
        for d in range(1, dim):
            k = k * count[d] + cells[:, d]
        return k

    key = key_of(c)
    order = torch.argsort(key)
    per_cell = torch.bincount(key, minlength=math.prod(count))
    first = torch.cumsum(per_cell, 0) - per_cell
    cs = c[order]
    starts, counts = [], []
    for o in _grid(*[range(-1, 2)] * dim).astype(int).tolist():
        nb = cs + torch.tensor(o, device=dev)
        if box is None:
            ok = ((nb >= 0) & (nb < lim)).all(dim=1)
            nb = torch.minimum(nb.clamp(min=0), lim - 1)
        else:
            ok = torch.ones(n, dtype=torch.bool, device=dev)
            nb = nb % lim
        k = key_of(nb)
        starts.append(first[k])
        counts.append(torch.where(ok, per_cell[k], 0))
    start, num = torch.stack(starts, 1), torch.stack(counts, 1)
    xs = x[order]
    upto = torch.cumsum(num.sum(dim=1), 0).cpu().numpy()
    size = 1 << 26 if dev.type == "cuda" else 1 << 22
    chunks, a = [], 0
    while a < n:
        done = int(upto[a - 1]) if a else 0
        b = max(a + 1, int(np.searchsorted(upto, done + size)))
        m = num[a:b].reshape(-1)
        rep = torch.repeat_interleave(torch.arange(m.numel(), device=dev), m)
        k = torch.arange(rep.numel(), device=dev) - (torch.cumsum(m, 0) - m)[rep]
        k += start[a:b].reshape(-1)[rep]
        p = a + torch.div(rep, num.shape[1], rounding_mode="floor")
        d = xs[p] - xs[k]
        if box is not None:
            size_t = torch.tensor(box, dtype=x.dtype, device=dev)
            d -= size_t * torch.round(d / size_t)
        r = torch.sqrt((d * d).sum(dim=1))
        near = (r <= h) & (p != k)
        chunks.append((order[p[near]], order[k[near]], d[near], r[near]))
        a = b
    return chunks


class _Exact:
    """One system of the inputs in FP64 torch tensors."""

    def __init__(self, s, device):
        def t(a):
            return torch.tensor(a, dtype=torch.float64, device=device)
        self.s, self.dim = s, s.dim
        self.x, self.v = t(s.x[:, :s.dim]), t(s.v[:, :s.dim])
        self.rho, self.P = t(s.rho), t(s.P)
        self.a = torch.zeros_like(self.x)
        self.fluid = t(s.type) == 0.0
        self.g = t(s.g[:s.dim])
        self.box = None if s.box is None else [float(b) for b in s.box]
        h = s.h
        if s.dim == 2:  # Wendland's quintic kernel and its derivative over r
            self.kW, self.kdW = s.m * 7 / math.pi / h ** 2, -s.m * 140 / math.pi / h ** 4
        else:
            self.kW, self.kdW = s.m * 10.5 / math.pi / h ** 3, -s.m * 210 / math.pi / h ** 5

    def build(self):
        if self.box is not None:
            self.x = self.x - torch.floor(self.x)
        self.near = _neighbours(self.x, self.s.h, self.box)

    def sum(self, term, shape):
        out = torch.zeros(shape, dtype=torch.float64, device=self.x.device)
        for p, q, d, r in self.near:
            out.index_add_(0, p, term(p, q, d, r))
        return out

    def density(self):
        def w(p, q, d, r):
            u = 1.0 - r / self.s.h
            return u ** 4 * (5.0 - 4.0 * u)
        return self.kW * (self.sum(w, self.rho.shape) + 1.0)

    def force(self):
        """internal_force! of the collapse program with Monaghan's viscosity."""
        s = self.s
        pr = self.P / self.rho ** 2

        def f(p, q, d, r):
            u3 = (1.0 - r / s.h) ** 3
            dv = self.v[p] - self.v[q]
            A = pr[p] + pr[q]
            if s.alpha:
                vx = (dv * d).sum(dim=1)
                rhobar = 0.5 * (self.rho[p] + self.rho[q])
                visc = -s.alpha * s.c * s.hs * vx / (rhobar * (r * r + 0.01 * s.hs ** 2))
                A = A + torch.where(vx < 0.0, visc, 0.0)
            t = -self.kdW * (u3 * A)[:, None] * d
            if s.mu:
                t = t + 2.0 * self.kdW * s.mu / s.rho0 ** 2 * u3[:, None] * dv
            return t
        return torch.where(self.fluid[:, None], self.sum(f, self.x.shape), 0.0)

    def kick(self, k):
        self.v = torch.where(self.fluid[:, None], self.v + k * (self.a + self.g), self.v)

    def move(self, k):
        self.x = torch.where(self.fluid[:, None], self.x + k * self.v, self.x)

    def wcsph(self, steps):
        s = self.s
        self.build()
        rho0 = self.density()
        for k in range(steps):
            if k:
                self.build()
            self.rho = self.density()
            self.P = s.c ** 2 * (self.rho - rho0)
            self.a = self.force()
            self.kick(s.dt)
            self.move(s.dt)

    def collapse(self, steps):
        s = self.s
        half = 0.5 * s.dt
        self.build()
        self.a = self.force()
        for _ in range(steps):
            self.kick(half)
            self.move(half)
            self.build()

            def rate(p, q, d, r):
                xv = (d * (self.v[p] - self.v[q])).sum(dim=1)
                return (1.0 - r / s.h) ** 3 * (xv + 2.0 * s.nu * (self.rho[p] - self.rho[q]))
            self.rho = self.rho + s.dt * self.kdW * self.sum(rate, self.rho.shape)
            self.P = s.c ** 2 * (self.rho - s.rho0)
            self.move(half)
            self.build()
            self.a = self.force()
            self.kick(half)

    def collide(self):
        """One step of the collision program; returns the energy after it."""
        s = self.s
        self.build()
        rho0 = self.density()

        def force():
            def f(p, q, d, r):
                A = (1.0 - r / s.h) ** 3 * (self.P[p] + self.P[q])
                return -self.kdW / s.rho0 ** 2 * A[:, None] * d
            return self.sum(f, self.x.shape)
        self.P = torch.zeros_like(rho0)
        self.v = self.v + 0.5 * s.dt * force()
        self.x = self.x + s.dt * self.v
        self.build()
        self.rho = self.density()
        self.P = s.c ** 2 * (self.rho - rho0)
        self.v = self.v + 0.5 * s.dt * force()
        kinetic = 0.5 * s.m * (self.v ** 2).sum()
        inner = 0.5 * s.m * s.c ** 2 / s.rho0 ** 2 * ((self.rho - rho0) ** 2).sum()
        return float(kinetic + inner)

    def full(self, a):
        out = torch.zeros((a.shape[0], 3), dtype=torch.float64, device=a.device)
        out[:, :self.dim] = a
        return out


def _exact_probes(case, s, seed, device):
    """Shepard denominators and velocity sums over the fluid at the points."""
    fluid = s.type == 0.0
    points = _probe_points(case, s, seed)
    n = len(points)
    x = torch.tensor(np.concatenate([points, s.x[fluid]]), device=device)
    v = torch.tensor(s.v[fluid], device=device)
    out = torch.zeros((n, 4), dtype=torch.float64, device=device)
    kW = s.m * 10.5 / math.pi / s.h ** 3
    for p, q, _, r in _neighbours(x, s.h, None):
        take = (p < n) & (q >= n)
        p, q, u = p[take], q[take] - n, 1.0 - r[take] / s.h
        w = kW * u ** 4 * (5.0 - 4.0 * u)
        out.index_add_(0, p, torch.cat([w[:, None], w[:, None] * v[q]], dim=1))
    return out


def exact(case, seed):
    dim = case.get("dim", 2)
    passes = case.get("steps", case.get("iterations", 1)) + 1
    if case["kind"] == "operators" or case.get("scheme") == "collapse_dry":
        passes *= 2
    cells = 3 ** dim * (4.8 if case["kind"] != "collision" else 2.4) ** dim
    if _particles(case) * cells * passes > EXACT_CANDIDATES:
        return None
    device = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    systems = _systems(case, seed)
    if case["kind"] == "probes":
        return _exact_probes(case, systems[0], seed, device)
    done, energy = [], None
    for s in systems:
        e = _Exact(s, device)
        if case["kind"] == "collision":
            energy = e.collide()
        elif case["kind"] == "operators":
            e.collapse(case["iterations"])
        elif case.get("scheme") == "collapse_dry":
            e.collapse(case["steps"])
        else:
            e.wcsph(case["steps"])
        done.append(e)
    out = dict(x=torch.cat([e.full(e.x) for e in done]), v=torch.cat([e.full(e.v) for e in done]),
               rho=torch.cat([e.rho for e in done]))
    if energy is not None:
        out["energy"] = energy
    return out
