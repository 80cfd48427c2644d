"""Timed cases of the engine_step path, each through the public Python entry points.

A case is what a simulation script does between two looks at its particles:
some steps in one call, then a read of the positions (and of the velocities
and species where the dynamics carry them).  The systems are those of the
repository's workloads: Morse cell sorting (overdamped), Morse + Lennard-Jones
mixtures, DPD droplets with a Fick flux, bonded chains, radius-dependent
potentials, DPD Couette flow between walls, Runge-Kutta 4, the replica
ensemble, and the force evaluation alone; in both precisions of the device,
with neighbour lists and without (the default), from a thousand particles to
two million.

Every table potential is handed over as its own record (intervals and
coefficients made here), so that exact() evaluates the same potential in
64 bits.  Mixed-precision results, which the device computes in FP32, are
returned as FP32 tensors, FP64 results as FP64.  Positions are returned
unwrapped against the initial ones, as for a mean-square displacement: a
particle near a periodic face is not at one side or the other by rounding.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    if "tissue_forge_amd" not in sys.modules:
        pkg = os.path.join(_ROOT, "tissue-forge_amd")
        spec = importlib.util.spec_from_file_location("tissue_forge_amd", os.path.join(pkg, "__init__.py"),
                                                      submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["tissue_forge_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["tissue_forge_amd"]


def listed():
    return [
        # a thousand cells in an interactive script: one step, a look at the
        # energies and positions, the next step
        dict(name="interactive_1k", kind="sort", n=1000, prec="mixed", skin=0.0, steps=1),
        # the cell-sorting example at its own size, in double precision
        dict(name="sort_8k_fp64_lists", kind="sort", n=8000, prec="fp64", skin=0.4, steps=100),
        # the same tissue four times larger with every setting at its default
        dict(name="sort_30k", kind="sort", n=30011, prec="mixed", skin=0.0, steps=20),
        # the large production run: two million particles of four types
        dict(name="mixture_2M_lists", kind="mixture", n=2_000_000, prec="mixed", skin=0.5, steps=50),
        # a mid-size run in double precision
        dict(name="mixture_300k_fp64_lists", kind="mixture", n=300_007, prec="fp64", skin=0.5, steps=25),
        # two DPD droplets exchanging a species
        dict(name="droplets_250k_lists", kind="droplets", n=250_000, prec="mixed", skin=0.4, steps=25),
        # a melt of 32-bead chains with bonds and angles
        dict(name="chains_1M_lists", kind="chains", n=1_000_000, prec="mixed", skin=0.6, steps=25),
        # cells of three sizes: potentials of the distance between surfaces
        dict(name="radii_100k", kind="radii", n=100_003, prec="mixed", skin=0.0, steps=10),
        # DPD fluid sheared between a resting and a moving wall
        dict(name="couette_24k", kind="couette", n=24_000, prec="mixed", skin=0.0, steps=25),
        # fourth-order integration of a Lennard-Jones fluid
        dict(name="rk4_64k", kind="rk4", n=64_000, prec="mixed", skin=0.0, steps=5),
        # a parameter sweep: replicas of the sorting experiment in one launch
        dict(name="sweep_48", kind="sweep", n=48, prec="mixed", skin=0.3, steps=20),
        # forces and energies of a given state (no update), as an external
        # integrator or an analysis asks for
        dict(name="forces_120k", kind="forces", n=120_000, prec="mixed", skin=0.0, steps=0),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same kinds: sizes over the ranges each kind is used at."""
    kind = rng.choice(["sort", "sort", "mixture", "mixture", "droplets", "chains", "radii", "couette", "rk4",
                       "sweep", "forces"])
    prec = "fp64" if rng.random() < 0.3 else "mixed"
    lists = rng.random() < 0.6
    if kind == "sort":
        n = _spread(rng, 800, 200_000)
        return dict(kind=kind, n=n, prec=prec, skin=round(rng.uniform(0.3, 0.5), 2) if lists else 0.0,
                    steps=rng.choice([1, 10, 40]))
    if kind == "mixture":
        n = _spread(rng, 5_000, 1_500_000)
        return dict(kind=kind, n=n, prec=prec, skin=round(rng.uniform(0.3, 0.6), 2) if lists else 0.0,
                    steps=rng.choice([5, 20]))
    if kind == "droplets":
        return dict(kind=kind, n=_spread(rng, 10_000, 600_000), prec=prec,
                    skin=round(rng.uniform(0.3, 0.5), 2) if lists else 0.0, steps=rng.choice([5, 20]))
    if kind == "chains":
        return dict(kind=kind, n=32 * _spread(rng, 200, 31_250), prec=prec,
                    skin=round(rng.uniform(0.4, 0.7), 2) if lists else 0.0, steps=rng.choice([5, 20]))
    if kind == "radii":
        return dict(kind=kind, n=_spread(rng, 2_000, 300_000), prec=prec, skin=0.0, steps=rng.choice([2, 10]))
    if kind == "couette":
        return dict(kind=kind, n=_spread(rng, 3_000, 200_000), prec=prec,
                    skin=round(rng.uniform(0.3, 0.5), 2) if lists else 0.0, steps=rng.choice([5, 20]))
    if kind == "rk4":
        return dict(kind=kind, n=_spread(rng, 5_000, 200_000), prec=prec, skin=0.0, steps=rng.choice([1, 4]))
    if kind == "sweep":
        return dict(kind=kind, n=rng.randint(5, 64), prec=prec, skin=0.3 if lists else 0.0, steps=rng.choice([5, 20]))
    return dict(kind="forces", n=_spread(rng, 1_000, 500_000), prec=prec, skin=0.0, steps=0)


# ---- potentials: piecewise-quintic records ------------------------------------------------------

_SCALED, _SHIFTED, _ANGLE = 1 << 11, 1 << 12, 1 << 6


def _table(fn, a, b, n, flags=0, r0p1=1.0):
    """The record of fn on [a, b]: n equal intervals, each a quintic through Chebyshev nodes."""
    width = (b - a) / n
    al1 = (1.0 - 1e-10) / width
    alpha = [1.0 - a * al1, al1, 0.0]
    nodes = np.cos((np.arange(6) + 0.5) * np.pi / 6)
    inv = np.linalg.inv(np.vander(nodes, 6))
    c = np.zeros((n + 1, 8))
    for k in range(n + 1):
        mid = a + (max(k, 1) - 0.5) * width
        c[k, 0], c[k, 1] = mid, 2.0 / width
        c[k, 2:] = inv @ fn(mid + 0.5 * width * nodes)
    return dict(kind="table", flags=flags, a=a, b=b, r0p1=r0p1, alpha=alpha, n=n, c=c)


def _morse(d, a, r0, lo, hi, flags=0, r0p1=1.0):
    return _table(lambda r: d * (np.exp(2 * a * (r0 - r)) - 2 * np.exp(a * (r0 - r))), lo, hi, 24, flags, r0p1)


def _lj(lo, hi):
    return _table(lambda r: 4.0 * (r ** -12 - r ** -6), lo, hi, 24)


def _dpd():
    return dict(kind="dpd", alpha=25.0, gamma=4.5, sigma=3.0, b=1.0)


# ---- systems --------------------------------------------------------------------------------------


def _lattice(rng, n, density, winding=False):
    """A jittered cubic lattice: no pair starts inside a repulsive core.  winding: every site next to the one before."""
    m = int(math.ceil(n ** (1.0 / 3.0) - 1e-9))
    a = density ** (-1.0 / 3.0)
    g = np.stack(np.meshgrid(np.arange(m), np.arange(m), np.arange(m), indexing="ij"), axis=-1)
    if winding:
        g[1::2] = g[1::2, ::-1].copy()
        line = np.arange(m * m).reshape(m, m) % 2 == 1
        g[line] = g[line][:, ::-1].copy()
    g = g.reshape(-1, 3)[:n]
    return np.mod((g + 0.5) * a + rng.uniform(-0.1 * a, 0.1 * a, size=(n, 3)), m * a), m * a


def _system(case, seed):
    """One system as plain values: box, types (mass, radius, overdamped), potentials, bindings, particles."""
    kind, n = case["kind"], case["n"]
    rng = np.random.default_rng(seed)
    s = dict(dim=None, cutoff=2.5, dt=0.005, types=[(40.0, 0.4, True)], pots=[], bind=[], x=None, v=None,
             ptype=np.zeros(n, dtype=np.int32), species=None, flux=0.0, bonds=None, angles=None, rk4=False,
             wall_speed=None)
    if kind == "sort":
        L = float(n) ** (1.0 / 3.0)
        while math.floor(L / (L / 3)) < 3:   # small boxes: three cells per axis
            L *= 1.0 + 1e-12
        rc = min(3.0, L / 3.0 * (1.0 - 1e-9))
        s.update(dim=[L] * 3, cutoff=rc, types=[(40.0, 0.4, True)] * 2, x=rng.uniform(0.0, L, size=(n, 3)),
                 ptype=(np.arange(n) % 2).astype(np.int32),
                 pots=[_morse(3.0, 5.0, 1.0, 0.5, rc), _morse(case.get("d_ab", 0.5), 5.0, 1.0, 0.5, rc)],
                 bind=[(0, 0, 0), (0, 1, 1), (1, 0, 1)])
    elif kind == "mixture":
        L = float(n) ** (1.0 / 3.0)
        s.update(dim=[L] * 3, types=[(40.0, 0.4, True)] * 4, x=rng.uniform(0.0, L, size=(n, 3)),
                 ptype=rng.integers(0, 4, size=n).astype(np.int32), pots=[_morse(3.0, 5.0, 1.0, 0.5, 2.5), _lj(0.8, 2.5)],
                 bind=[(0, t, t) for t in range(4)] + [(1, a, b) for a in range(4) for b in range(a + 1, 4)])
    elif kind in ("droplets", "couette"):
        if kind == "droplets":
            L = (n / 3.0) ** (1.0 / 3.0)
            dim = [L] * 3
        else:
            L = (n / 1.5) ** (1.0 / 3.0)
            dim = [L, L, 0.5 * L]
        x = rng.uniform(0.0, 1.0, size=(n, 3)) * dim
        s.update(dim=dim, cutoff=1.0, dt=0.01, types=[(1.0, 0.5, False)], pots=[_dpd()], bind=[(0, 0, 0)], x=x,
                 v=np.zeros((n, 3)))
        if kind == "droplets":
            r = min(10.0, L / 4 - 1e-9)
            drop = [np.sum((x - [c * L, L / 2, L / 2]) ** 2, axis=1) < r * r for c in (0.25, 0.75)]
            s["types"] = [(1.0, 0.5, False)] * 3
            s["bind"] = [(0, a, b) for a in range(3) for b in range(a, 3)]
            s["species"] = np.full((n, 1), 0.5)
            s["flux"] = 0.1
            for k, inside in enumerate(drop):
                s["ptype"][inside] = k + 1
                s["v"][inside, 0] = 1.0 - 2.0 * k
                s["species"][inside, 0] = float(k)
        else:
            s["wall_speed"] = 1.0
    elif kind == "chains":
        # beads along a line that winds through a jittered lattice, cut into chains of 32
        x, L = _lattice(rng, n, 0.8, winding=True)
        ids = np.arange(n, dtype=np.int32).reshape(n // 32, 32)
        s.update(dim=[L] * 3, dt=0.002, types=[(1.0, 0.5, False)], bind=[(0, 0, 0)], x=x, v=rng.normal(size=(n, 3)),
                 pots=[_lj(0.8, 2.5), _table(lambda r: 50.0 * (r - 1.0) ** 2, 0.0, 2.0, 1),
                       _table(lambda c: 10.0 * (np.arccos(np.clip(c, -1.0, 1.0)) - math.pi) ** 2, -1.0, 1.0, 58, _ANGLE)],
                 bonds=(1, np.stack([ids[:, :-1].ravel(), ids[:, 1:].ravel()], axis=1)),
                 angles=(2, np.stack([ids[:, :-2].ravel(), ids[:, 1:-1].ravel(), ids[:, 2:].ravel()], axis=1)))
    elif kind == "radii":
        x, L = _lattice(rng, n, 0.5)
        s.update(dim=[L] * 3, dt=0.002, types=[(1.0 + t, r, False) for t, r in enumerate((0.3, 0.45, 0.6))], x=x,
                 v=rng.normal(size=(n, 3)), ptype=rng.integers(0, 3, size=n).astype(np.int32),
                 pots=[_morse(1.0, 6.0, 1.0, 1.0, 4.0, _SHIFTED, 1.0), _morse(0.5, 3.0, 1.0, 0.5, 3.0, _SCALED)],
                 bind=[(0, 0, 0), (0, 0, 1), (1, 1, 1), (1, 1, 2), (1, 2, 2), (1, 0, 2)])
    elif kind == "rk4":
        x, L = _lattice(rng, n, 0.7)
        s.update(dim=[L] * 3, dt=0.002, types=[(1.0, 0.5, False)], x=x, v=rng.normal(size=(n, 3)), rk4=True,
                 pots=[_lj(0.7, 2.5)], bind=[(0, 0, 0)])
    else:   # forces: a Lennard-Jones and Morse mixture as it stands
        x, L = _lattice(rng, n, 1.0)
        s.update(dim=[L] * 3, x=x, types=[(40.0, 0.4, True)] * 4, ptype=rng.integers(0, 4, size=n).astype(np.int32),
                 pots=[_morse(3.0, 5.0, 1.0, 0.5, 2.5), _lj(0.8, 2.5)],
                 bind=[(0, t, t) for t in range(4)] + [(1, a, b) for a in range(4) for b in range(a + 1, 4)])
    return s


def _systems(case, seed):
    if case["kind"] != "sweep":
        return [_system(case, seed)]
    rng = np.random.default_rng(5)   # the sweep's sizes and strengths; the particles are the seed's
    out = []
    for r in range(case["n"]):
        n = int(round(math.exp(rng.uniform(math.log(500), math.log(20_000)))))
        out.append(_system(dict(kind="sort", n=n, d_ab=float(rng.uniform(0.2, 2.0))), 1000 * seed + r + 1))
    return out


def _grid(s):
    return [max(3, int(math.floor(d / s["cutoff"]))) for d in s["dim"]]


def _engine(s, skin):
    tf = _package()
    eng = tf.Engine(dim=s["dim"], cells=_grid(s), cutoff=s["cutoff"], dt=s["dt"], nspecies=0 if s["species"] is None else 1,
                    integrator=tf.RUNGE_KUTTA_4 if s["rk4"] else tf.FORWARD_EULER)
    for k, (mass, radius, over) in enumerate(s["types"]):
        eng.add_type("T%d" % k, mass=mass, radius=radius, dynamics=tf.OVERDAMPED if over else tf.NEWTONIAN)
    pots = []
    for p in s["pots"]:
        if p["kind"] == "dpd":
            pots.append(tf.Potential.dpd(alpha=p["alpha"], gamma=p["gamma"], sigma=p["sigma"], cutoff=p["b"]))
        else:
            pots.append(tf.Potential.from_table(p["flags"], p["a"], p["b"], p["r0p1"], p["alpha"], p["n"], p["c"]))
    for p, a, b in s["bind"]:
        eng.bind(pots[p], a, b)
    if s["flux"]:
        nt = len(s["types"])
        for a in range(nt):
            for b in range(a, nt):
                eng.add_flux(tf.FLUX_FICK, a, b, 0, 0, s["flux"])
    if s["wall_speed"] is not None:
        eng.set_boundary("bottom", tf.BOUNDARY_NO_SLIP)
        eng.set_boundary("top", tf.BOUNDARY_VELOCITY, velocity=(s["wall_speed"], 0.0, 0.0))
    if skin:
        eng.set_verlet(skin)
    eng.add_particles(s["ptype"], s["x"], s["v"], s["species"])
    if s["bonds"] is not None:
        eng.add_bonds(pots[s["bonds"][0]], s["bonds"][1])
        eng.add_angles(pots[s["angles"][0]], s["angles"][1])
    return eng


def prepare(case, seed):
    """The engines on the device, and what unwrapping needs: initial positions, box edges, one buffer."""
    tf = _package()
    systems = _systems(case, seed)
    engines = [_engine(s, case["skin"]) for s in systems]
    prec = tf.PREC_FP64 if case["prec"] == "fp64" else tf.PREC_MIXED
    st = dict(case=case, engines=engines, ensemble=None, dtype=torch.float64 if case["prec"] == "fp64" else torch.float32)
    if case["kind"] == "sweep":
        st["ensemble"] = tf.Ensemble(engines, prec)
    else:
        engines[0].to_device(prec)
    st["x0"] = [torch.from_numpy(s["x"]) for s in systems]
    st["box"] = [_edges(s, "cpu") for s in systems]
    st["buf"] = [torch.empty_like(x) for x in st["x0"]]
    return st


def _edges(s, device):
    """Period of each axis (0: not periodic)."""
    return torch.tensor([0.0 if s["wall_speed"] is not None and k == 2 else s["dim"][k] for k in range(3)],
                        dtype=torch.float64, device=device)


def _unwrap(x, x0, box, buf):
    """x moved by whole periods to within half a period of x0, in place."""
    torch.sub(x, x0, out=buf)
    buf.mul_(torch.where(box > 0, 1.0 / box, 0.0)).round_()
    return x.addcmul_(buf, box, value=-1.0)


def _positions(st, k):
    x = torch.from_numpy(st["engines"][k].positions())
    return _unwrap(x, st["x0"][k], st["box"][k], st["buf"][k]).to(st["dtype"])


def run(st):
    case, eng = st["case"], st["engines"][0]
    if case["kind"] == "forces":
        eng.force()
        e = eng.energies()
        return dict(f=torch.from_numpy(eng.particles()["f"]).to(st["dtype"]),
                    e=torch.tensor([e["epot"], e["virial"]], dtype=st["dtype"]))
    if case["kind"] == "sweep":
        st["ensemble"].step(case["steps"])
        return dict(x=torch.cat([_positions(st, k) for k in range(len(st["engines"]))]))
    eng.step(case["steps"])
    out = dict(x=_positions(st, 0))
    if case["kind"] == "sort" and case["steps"] == 1:
        e = eng.energies()
        out["e"] = torch.tensor([e["epot"], e["virial"]], dtype=st["dtype"])
    if case["kind"] not in ("sort", "mixture"):
        p = eng.particles()
        out["v"] = torch.from_numpy(p["v"]).to(st["dtype"])
        if case["kind"] == "droplets":
            out["species"] = torch.from_numpy(p["species"]).to(st["dtype"])
    return out


def work(case):
    """State read and written once and outputs written once; every pair in range evaluated once per force evaluation."""
    per_pair = dict(droplets=45, couette=40).get(case["kind"], 40)
    n, rc, rho = case["n"], 2.5, 1.0
    if case["kind"] == "sweep":
        n, rc = int(case["n"] * (20_000 - 500) / math.log(40.0)), 3.0
    elif case["kind"] == "sort":
        rc = min(3.0, n ** (1.0 / 3.0) / 3.0)
    elif case["kind"] in ("droplets", "couette"):
        rc, rho = 1.0, 3.0
    elif case["kind"] in ("chains", "radii", "rk4"):
        rho = dict(chains=0.8, radii=0.5, rk4=0.7)[case["kind"]]
    word = 8 if case["prec"] == "fp64" else 4
    values = dict(sort=3, mixture=3, sweep=3, droplets=7, forces=4).get(case["kind"], 6)
    evals = 1 if case["kind"] == "forces" else case["steps"] * (4 if case["kind"] == "rk4" else 1)
    pairs = 0.5 * n * rho * 4.0 / 3.0 * math.pi * rc ** 3
    return dict(bytes=float(n * (2 * 7 * word + values * word)), flops=float(evals * (pairs * per_pair + n * 20)))


# ---- the same passes in 64 bits, in plain torch ------------------------------------------------


def _half_stencil():
    return [(0, 0, 0)] + [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1) if (a, b, c) > (0, 0, 0)]


class _Plain:
    """One system in 64-bit torch: every pair within the cutoff once, found through cells of at least the cutoff."""

    def __init__(self, s, device):
        self.s, self.dev = s, device

        def put(a):
            return torch.as_tensor(np.asarray(a), device=device)

        self.x = put(s["x"]).clone()
        self.n = self.x.shape[0]
        self.v = torch.zeros_like(self.x) if s["v"] is None else put(s["v"]).clone()
        self.t = put(s["ptype"]).long()
        self.nt = len(s["types"])
        self.mass = put(np.array([t[0] for t in s["types"]], dtype=np.float64))[self.t]
        self.im = (1.0 / self.mass)[:, None]
        self.radius = put(np.array([t[1] for t in s["types"]], dtype=np.float64))[self.t]
        self.over = s["types"][0][2]
        self.dim = torch.tensor(s["dim"], dtype=torch.float64, device=device)
        self.m = [int(math.floor(d / (d / c))) for d, c in zip(s["dim"], _grid(s))]   # the engine's own cells
        self.h = self.dim / torch.tensor(self.m, dtype=torch.float64, device=device)
        self.period = _edges(s, device)
        self.sp = None if s["species"] is None else put(s["species"]).clone()[:, 0]
        self.q = torch.zeros(self.n, dtype=torch.float64, device=device)
        self.maps = torch.zeros(self.nt * self.nt, dtype=torch.long, device=device)
        for p, a, b in s["bind"]:
            self.maps[a * self.nt + b] = self.maps[b * self.nt + a] = p
        self.tables = [None if p["kind"] == "dpd" else put(p["c"]) for p in s["pots"]]

    def cells(self, x):
        m = torch.tensor(self.m, device=self.dev)
        return torch.minimum((x / self.h).floor().long().clamp_(min=0), m - 1)

    def image(self, d):
        inv = torch.where(self.period > 0, 1.0 / self.period, 0.0)
        return d - self.period * (d * inv).round()

    def table(self, p, r):
        """Energy and derivative of table p at r (clamped to its left end)."""
        pot, c = self.s["pots"][p], self.tables[p]
        r = r.clamp(min=pot["a"])
        k = (pot["alpha"][0] + pot["alpha"][1] * r).long().clamp_(1, pot["n"])
        row = c[k]
        u = (r - row[:, 0]) * row[:, 1]
        e, d = row[:, 2] * u + row[:, 3], row[:, 2]
        for j in range(4, 8):
            d = d * u + e
            e = e * u + row[:, j]
        return e, d * row[:, 1]

    def pair_terms(self, i, j, dx, r, f, out):
        """Adds the terms of the pairs (i, j) to f and to the energy, virial and pending flux."""
        s = self.s
        pot = self.maps[self.t[i] * self.nt + self.t[j]]
        over_r = torch.zeros_like(r)   # (force on i along dx) / r
        for p, rec in enumerate(s["pots"]):
            if rec["kind"] == "dpd":
                e = dx / r[:, None]
                ev = (e * (self.v[i] - self.v[j])).sum(1)
                om = 1.0 - r / rec["b"]
                fr = rec["alpha"] * om - rec["gamma"] * om * om * ev + rec["sigma"] * om / math.sqrt(s["dt"])
                over_r += torch.where((pot == p) & (r <= rec["b"]), fr / r, 0.0)
                continue
            sel = (pot == p).nonzero()[:, 0]
            if sel.numel() == 0 or rec["flags"] & _ANGLE:
                continue
            rr = r[sel]
            rt = rr
            if rec["flags"] & _SCALED:
                rt = rr / (self.radius[i[sel]] + self.radius[j[sel]])
            elif rec["flags"] & _SHIFTED:
                rt = rr - (self.radius[i[sel]] + self.radius[j[sel]]) + rec["r0p1"]
            e, d = self.table(p, rt)
            inside = rt <= rec["b"]
            over_r[sel] = torch.where(inside, -d / rr, 0.0)
            out["epot"] += float(torch.where(inside, e, 0.0).sum())
        f3 = over_r[:, None] * dx
        f.index_add_(0, i, f3)
        f.index_add_(0, j, f3, alpha=-1.0)
        out["virial"] += float((over_r * r * r).sum())
        if s["flux"]:
            qv = s["flux"] * (self.sp[i] - self.sp[j]) * (1.0 - r / s["cutoff"]) ** 2
            self.q.index_add_(0, i, qv, alpha=-1.0)
            self.q.index_add_(0, j, qv)
        if out.get("nd") is not None:
            w = 1.0 / (math.pi * s["cutoff"] ** 3)
            u = r / s["cutoff"]
            w = w * (1.0 - 1.5 * u * u + 0.75 * u ** 3)
            out["nd"].index_add_(0, i, w)
            out["nd"].index_add_(0, j, w)

    def forces(self, nd=False):
        rc, m = self.s["cutoff"], self.m
        out = dict(epot=0.0, virial=0.0, nd=None)
        if nd:
            out["nd"] = torch.full((self.n,), 1.0 / (math.pi * rc ** 3), dtype=torch.float64, device=self.dev)
        f = torch.zeros_like(self.x)
        loc = self.cells(self.x)
        cid = (loc[:, 0] * m[1] + loc[:, 1]) * m[2] + loc[:, 2]
        order = torch.argsort(cid)
        count = torch.bincount(cid, minlength=m[0] * m[1] * m[2])
        start = torch.cumsum(count, 0) - count
        mt = torch.tensor(m, device=self.dev)
        for sh in _half_stencil():
            o = torch.tensor(sh, device=self.dev)
            nb = loc + o
            ok = ((nb >= 0) & (nb < mt) | (self.period > 0)).all(1)
            nb = torch.remainder(nb, mt)
            nc = (nb[:, 0] * m[1] + nb[:, 1]) * m[2] + nb[:, 2]
            k = torch.where(ok, count[nc], 0)
            i = torch.repeat_interleave(torch.arange(self.n, device=self.dev), k)
            at = torch.arange(i.numel(), device=self.dev) - (torch.cumsum(k, 0) - k)[i]
            j = order[start[nc[i]] + at]
            del at
            if sh == (0, 0, 0):
                keep = i < j
                i, j = i[keep], j[keep]
            dx = self.image(self.x[i] - self.x[j])
            r2 = (dx * dx).sum(1)
            keep = r2 <= rc * rc
            self.pair_terms(i[keep], j[keep], dx[keep], r2[keep].sqrt(), f, out)
        self.bonded(f)
        return f, out

    def bonded(self, f):
        s = self.s
        if s["bonds"] is None:
            return
        p, ij = s["bonds"]
        i, j = torch.as_tensor(ij, device=self.dev).long().unbind(1)
        dx = self.image(self.x[i] - self.x[j])
        r = dx.norm(dim=1)
        _, d = self.table(p, r)
        f3 = torch.where(r <= s["pots"][p]["b"], -d / r, 0.0)[:, None] * dx
        f.index_add_(0, i, f3)
        f.index_add_(0, j, f3, alpha=-1.0)
        p, ijk = s["angles"]
        i, j, k = torch.as_tensor(ijk, device=self.dev).long().unbind(1)
        a, b = self.image(self.x[i] - self.x[j]), self.image(self.x[k] - self.x[j])
        ia, ib = 1.0 / a.norm(dim=1, keepdim=True), 1.0 / b.norm(dim=1, keepdim=True)
        c = (a * b).sum(1, keepdim=True) * ia * ib
        _, d = self.table(p, c[:, 0].clamp(-1.0, 1.0))
        fi = -d[:, None] * (b * ib - c * a * ia) * ia
        fk = -d[:, None] * (a * ia - c * b * ib) * ib
        f.index_add_(0, i, fi)
        f.index_add_(0, k, fk)
        f.index_add_(0, j, fi + fk, alpha=-1.0)

    def wrap(self):
        for k in range(3):
            if float(self.period[k]) > 0:
                self.x[:, k] = torch.remainder(self.x[:, k], self.dim[k])

    def step(self):
        s, dt = self.s, self.s["dt"]
        if s["rk4"]:
            p0, v0 = self.x.clone(), self.v.clone()
            sx, sv = torch.zeros_like(p0), torch.zeros_like(p0)
            vk = None
            for st, (wt, back, to) in enumerate(((1, 0.0, 0.5), (2, 0.5, 0.5), (2, 0.5, 1.0), (1, 1.0, 0.0))):
                f, _ = self.forces()
                xk = v0 if st == 0 else v0 + back * dt * vk
                vk = f * self.im
                sx += wt * xk
                sv += wt * vk
                self.x = p0 + (to * dt * xk if st < 3 else dt / 6.0 * sx)
                self.wrap()
            self.v = v0 + dt / 6.0 * sv
            return dict(epot=0.0, virial=0.0)
        f, out = self.forces()
        most = 0.05 * self.h
        if self.over:
            d = torch.minimum(torch.maximum(dt * f * self.im, -most), most)
            self.v = d / dt
        else:
            self.v = torch.minimum(torch.maximum(self.v + dt * f * self.im, -most / dt), most / dt)
            d = dt * self.v
        before = self.cells(self.x)
        self.x = self.x + d
        if s["wall_speed"] is not None:
            z, top = self.x[:, 2], float(self.dim[2])
            lo, hi = z < 0, z >= top
            self.x[:, 2] = torch.where(lo, -z, torch.where(hi, 2 * top - z, z))
            wall = torch.tensor([s["wall_speed"], 0.0, 0.0], dtype=torch.float64, device=self.dev)
            self.v = torch.where(lo[:, None], -self.v, torch.where(hi[:, None], 2 * wall - self.v, self.v))
        self.wrap()
        if self.sp is not None:   # a particle that changes cell keeps its pending flux for the next step
            stays = (self.cells(self.x) == before).all(1)
            self.sp = torch.where(stays, (self.sp + dt * self.q).clamp(min=0.0), self.sp)
            self.q = torch.where(stays, 0.0, self.q)
        return out


def exact(case, seed):
    """run()'s outputs after one pass from the prepared state, in 64 bits."""
    if case["kind"] == "sweep" and case["n"] * case["steps"] > 1000:
        return None   # one small system after another takes plain torch too long
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    outs = []
    for s in _systems(case, seed):
        p = _Plain(s, dev)
        x0 = p.x.clone()
        if case["kind"] == "forces":
            f, e = p.forces(nd=True)
            return dict(f=torch.cat([f, e["nd"][:, None]], dim=1).cpu(),
                        e=torch.tensor([e["epot"], e["virial"]], dtype=torch.float64))
        for _ in range(case["steps"]):
            e = p.step()
        o = dict(x=_unwrap(p.x, x0, p.period, torch.empty_like(x0)).cpu())
        if case["kind"] not in ("sort", "mixture", "sweep"):
            o["v"] = p.v.cpu()
        if case["kind"] == "droplets":
            o["species"] = p.sp.cpu()[:, None]
        if case["kind"] == "sort" and case["steps"] == 1:
            o["e"] = torch.tensor([e["epot"], e["virial"]], dtype=torch.float64)
        outs.append(o)
    if case["kind"] == "sweep":
        return dict(x=torch.cat([o["x"] for o in outs]))
    return outs[0]
