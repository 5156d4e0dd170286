"""The work that users of this library have it do, as timed cases.

Each case is a piece of a real program through the public entry points
(`particlebase_amd.System`): the loops of the reference's drivers and of this
repository's benchmark, with a trajectory snapshot (`System.get`) at the end
of every pass, as a program that writes dumps takes one.  `listed()` holds the
fixed cases, `draw(rng)` others of the same ranges:

    force    one LJ force + energy evaluation (cudaParticleMD::calcForce)
    run      the fused LJ loop of one system (FP64 or mixed precision)
    batch    the fused LJ loop of many independent replicas in one launch
    nlist    the neighbour-list MD loop (makeNList every 10 steps)
    gauss    the isokinetic MD loop (calcForce + GaussianThermo)
    gr       radial distribution histograms of a batch of replicas
    sph      the dam-break loop, reference physics (Lucy) or the weakly
             compressible one (M4 spline, Tait, artificial viscosity)
    dem      the granular loop, Hertz or linear spring-dashpot contacts, a
             settled bed (about 6 contacts a sphere) or a falling suspension

`exact(case, seed)` restates each in plain FP64 torch.
"""
import math

import numpy as np
import torch

import particlebase_amd as pb
from particlebase_amd import workloads

DT = 0.005            # LJ time step
RC = 2.5              # LJ cutoff, the benchmark's
SKIN = 0.3
THICKNESS = 0.5       # of the neighbour list that is made every 10 steps
KBT = 0.72
# sigma and epsilon of the two-species gas driver, relative to its first species
TWO_TYPES = [1.0, 1.0, 1.0346, 1.3427, 1.0346, 1.3427, 1.0692, 1.1680]

_context = []


def context():
    """One context for the process, as a program keeps it."""
    if not _context:
        _context.append(pb.Context(0))
    return _context[0]


# ------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest call a driver makes: one FP64 force and energy of 864 atoms
        {"name": "force_864", "kind": "force", "n": 864, "rho": 0.8442, "types": 1, "mixed": False},
        # the benchmark's small system: 4000 atoms, energies every 10 steps
        {"name": "run_4000_mixed", "kind": "run", "n": 4000, "rho": 0.8442, "types": 1,
         "mixed": True, "steps": 100, "every": 10},
        # an ordinary FP64 production run, a count that fills no tile evenly
        {"name": "run_107999_fp64", "kind": "run", "n": 107999, "rho": 0.8442, "types": 1,
         "mixed": False, "steps": 100, "every": 10},
        # the headline workload, a snapshot every 100 steps
        {"name": "run_1048576_mixed", "kind": "run", "n": 1048576, "rho": 0.8442, "types": 1,
         "mixed": True, "steps": 100, "every": 10},
        # the batched workload: 256 replicas of 500 to 20000 atoms
        {"name": "batch_256_mixed", "kind": "batch", "nrep": 256, "nmin": 500, "nmax": 20000,
         "mixed": True, "steps": 50, "every": 0},
        # the neighbour-list driver's loop on a two-species fluid
        {"name": "nlist_32000", "kind": "nlist", "n": 32000, "rho": 0.7, "types": 2, "steps": 20},
        # the isokinetic driver's loop at its own size (a 60 A box of argon)
        {"name": "gauss_4924", "kind": "gauss", "n": 4924, "rho": 0.8442, "types": 1, "steps": 20},
        # g(r) of the batched workload, 200 bins to half the box
        {"name": "gr_256", "kind": "gr", "nrep": 256, "nmin": 500, "nmax": 20000, "bins": 200},
        # the dam break at full size, reference physics
        {"name": "sph_lucy_796176", "kind": "sph", "physics": "lucy", "dx": 0.4 / 63, "steps": 20},
        # the dam break at a sixth of that, weakly compressible physics, odd spacing
        {"name": "sph_wc_133904", "kind": "sph", "physics": "wc", "dx": 0.4 / 31, "steps": 20},
        # the granular settle at full size: falling, few contacts, linear law
        {"name": "dem_linear_200000", "kind": "dem", "law": "linear", "bed": False, "n": 200000,
         "steps": 20},
        # a settled bed under the reference's Hertz law
        {"name": "dem_hertz_bed_60000", "kind": "dem", "law": "hertz", "bed": True, "n": 60000,
         "steps": 20},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["force", "run", "run", "batch", "nlist", "gauss", "gr", "sph", "sph", "dem",
                       "dem"])
    if kind == "force":
        return {"kind": kind, "n": int(_log(rng, 500, 300000)), "rho": rng.uniform(0.6, 0.9),
                "types": rng.choice([1, 1, 2]), "mixed": rng.random() < 0.5}
    if kind == "run":
        n = int(_log(rng, 800, 800000))
        return {"kind": kind, "n": n, "rho": rng.uniform(0.65, 0.9), "types": rng.choice([1, 1, 2]),
                "mixed": rng.random() < 0.5, "steps": rng.randint(50, 100),
                "every": rng.choice([1, 10, 25])}
    if kind == "batch":
        return {"kind": kind, "nrep": int(_log(rng, 3, 256)), "nmin": 500,
                "nmax": int(_log(rng, 1000, 20000)), "mixed": rng.random() < 0.7,
                "steps": rng.randint(20, 50), "every": rng.choice([0, 10])}
    if kind == "nlist":
        return {"kind": kind, "n": int(_log(rng, 2000, 120000)), "rho": rng.uniform(0.4, 0.85),
                "types": rng.choice([1, 2]), "steps": rng.randint(10, 30)}
    if kind == "gauss":
        return {"kind": kind, "n": int(_log(rng, 1000, 60000)), "rho": rng.uniform(0.7, 0.86),
                "types": 1, "steps": rng.randint(10, 30)}
    if kind == "gr":
        return {"kind": kind, "nrep": int(_log(rng, 1, 256)), "nmin": 500,
                "nmax": int(_log(rng, 1000, 20000)), "bins": rng.choice([50, 127, 200, 333, 400])}
    if kind == "sph":
        return {"kind": kind, "physics": rng.choice(["lucy", "wc"]),
                "dx": 0.4 / rng.uniform(8.0, 55.0), "steps": rng.randint(10, 20)}
    return {"kind": "dem", "law": rng.choice(["linear", "hertz"]), "bed": rng.random() < 0.6,
            "n": int(_log(rng, 2000, 200000)), "steps": rng.randint(10, 20)}


# ------------------------------------------------------------------ inputs
def _fluid(case, seed):
    """An LJ fluid a little off its lattice, with thermal velocities."""
    n = case["n"]
    w = workloads.lj_fcc(int(math.ceil((n / 4.0) ** (1.0 / 3.0) - 1e-12)), case["rho"], KBT,
                         seed=seed, natoms=n)
    w.r = w.r + 0.05 * workloads.normals(seed + 1000, 3 * n).reshape(n, 3)
    if case.get("types", 1) == 2:
        w.type = (workloads.uniform53(seed + 2000, n) < 0.8).astype(np.uint32)
        w.sigma_eps = np.array(TWO_TYPES)
    return w


def _replicas(case, seed):
    """The batched workload's sizes, densities and temperatures; positions off
    their lattice and velocities from the seed."""
    b = workloads.lj_replicas(case["nrep"], case["nmin"], case["nmax"], seed=5)
    for k, s in enumerate(b.systems):
        s.r = s.r + 0.05 * workloads.normals(seed + 5000 + k, 3 * s.n).reshape(s.n, 3)
        s.v = workloads.mb_velocities(s.n, s.T, s.m, seed + 10000 + k)
    return b


def _dam(case, seed):
    make = workloads.sph_dam_break if case["physics"] == "lucy" else workloads.sph_dam_break_config
    return make(case["dx"], jitter=0.2, seed=seed)


def _grains(case, seed):
    """Spheres of about a millimetre in a 0.1 m box: a bed of touching spheres
    (nearly equal radii on a pitch just below their diameter) or the settle
    workload's dispersed start; small random velocities."""
    n = case["n"]
    if case["bed"]:
        w = workloads.dem_settle(n, rmin=0.9999e-3, rmax=1.0e-3, gap=-2.5e-4, seed=seed, fill="bottom")
        vscale = 1.0e-3
    else:
        w = workloads.dem_settle(n, seed=seed)
        vscale = 0.05
    w.v = vscale * workloads.normals(seed + 3, 3 * n).reshape(n, 3)
    return w


DEM_LINEAR = {"kn": 1.0e4, "e": 0.8, "kt": 2.0e4 / 7.0, "mu": 0.5}
DEM_HERTZ = {"E": 2.11e9, "mu": 0.5, "sigma": 0.29,
             "gamma": -2.0 * math.log(0.8) / math.sqrt(math.pi ** 2 + math.log(0.8) ** 2),
             "mu_r": 0.1}


def _dem_dt(case):
    if case["bed"]:
        return 1.0e-6 if case["law"] == "linear" else 2.5e-7
    return 5.65685e-6 if case["law"] == "linear" else 5.0e-7


def _lj_system(w, counts=None, cells=None):
    s = pb.System(context(), [w.n] if counts is None else counts)
    s.set_cell(w.cell if cells is None else cells)
    return s


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case)
    if kind in ("force", "run", "nlist", "gauss"):
        w = _fluid(case, seed)
        s = _lj_system(w)
        s.import_particles(w.r, w.m, v=w.v, type=w.type)
        s.lj_set_params(w.sigma_eps, case["types"])
        s.lj_set_cutoff(RC * RC, shifted=True)
        s.clear_force(True)
        if kind == "nlist":
            s.setup_cells(RC + THICKNESS, periodic=True)
        elif kind == "gauss":
            s.setup_cells(RC, periodic=True)
    elif kind in ("batch", "gr"):
        b = _replicas(case, seed)
        r, v, m, t, cells = b.concat()
        s = _lj_system(None, b.counts, cells)
        s.import_particles(r, m, v=v, type=t)
        s.lj_set_params([1.0, 1.0], 1)
        s.lj_set_cutoff(RC * RC, shifted=True)
        s.clear_force(True)
        if kind == "gr":
            st["rstep"] = np.array([np.float32(x.L / (2.0 * case["bins"])) for x in b.systems])
    elif kind == "sph":
        w = _dam(case, seed)
        s = _lj_system(w)
        s.import_particles(w.r, w.m, is_fixed=w.fixed)
        if case["physics"] == "lucy":
            s.sph_set_properties(w.mu0, w.c, w.h)
            support = w.h
        else:
            s.sph_set_wcsph(w.h, w.rho0, w.c[0], 7.0, 0.1, 0.0)
            support = 2 * w.h
        s.setup_cells(support, periodic=False)
        st["dt"] = 0.25 * w.h / float(w.c[0])
        st["vlim"] = 2 * support / st["dt"]
    else:
        w = _grains(case, seed)
        s = _lj_system(w)
        s.import_particles(w.r, w.m, v=w.v, is_fixed=w.fixed)
        if case["law"] == "linear":
            s.dem_set_linear(DEM_LINEAR["kn"], DEM_LINEAR["e"], DEM_LINEAR["kt"], DEM_LINEAR["mu"],
                             w.rad)
        else:
            s.dem_set_properties(DEM_HERTZ["E"], DEM_HERTZ["mu"], DEM_HERTZ["sigma"],
                                 DEM_HERTZ["gamma"], DEM_HERTZ["mu_r"], w.rad)
        s.rot_set_inertia(w.rad)
        s.setup_cells(2 * float(w.rad.max()), periodic=False)
        st["dt"] = _dem_dt(case)
        st["vlim"] = 2 * 0.9e-3 / st["dt"]
    context().sync()
    st["s"] = s
    return st


# -------------------------------------------------------------------- runs
def _energies(e, mixed):
    # energies of the mixed form are sums of FP32 pair terms: FP32 numbers
    return e.astype(np.float32) if mixed else e


def run(st):
    s, kind = st["s"], st["kind"]
    if kind == "force":
        pe, w = s.lj_force(pb.PB_MIXED if st["mixed"] else pb.PB_FP64, energies=True)
        return {"pe": _energies(pe, st["mixed"]), "w": _energies(w, st["mixed"]), "F": s.get("F")}
    if kind in ("run", "batch"):
        e, _ = s.lj_run(DT, st["steps"], precision=pb.PB_MIXED if st["mixed"] else pb.PB_FP64,
                        skin=SKIN, rebuild_every=20, energy_every=st["every"])
        out = {"r": s.get("r"), "v": s.get("v")}
        if st["every"]:
            out["e"] = _energies(e, st["mixed"])
        return out
    if kind == "nlist":
        rt2 = (RC + THICKNESS - 1e-3) ** 2
        pe = []
        for k in range(st["steps"]):
            if k % 10 == 0:
                s.bin()
                s.nlist_build(rt2)
            pe.append(s.lj_force_nlist())
            s.vv_step(DT)
            s.treat_periodic()
        return {"r": s.get("r"), "v": s.get("v"), "pe_w": np.array(pe)}
    if kind == "gauss":
        t = []
        for _ in range(st["steps"]):
            s.bin()
            s.lj_force(pb.PB_FP64, energies=True)
            t.append(s.mv2()[0])
            s.gt_step(DT, 1e-10)
            s.treat_periodic()
        return {"r": s.get("r"), "v": s.get("v"), "mv2": np.array(t)}
    if kind == "gr":
        return s.gr_hist(st["rstep"], st["bins"]).astype(np.int64)
    if kind == "sph":
        dt = st["dt"]
        for _ in range(st["steps"]):
            s.bin()
            s.sph_density()
            s.sph_acceleration()
            s.add_acceleration(2, -9.81)
            s.lf_step(dt)
            s.inspect_velocity(st["vlim"], 0.04, 0.0025)
            s.treat_absolute()
        return {"r": s.get("r"), "v": s.get("v"), "num": s.get("sph_num")}
    dt = st["dt"]
    nnz = []
    for _ in range(st["steps"]):
        s.bin()
        nnz.append(s.dem_calc_force(dt, autotune=True))
        s.calc_acceleration()
        s.add_acceleration(2, -9.8)
        s.lf_step(dt)
        s.rot_step(dt)
        s.inspect_velocity(st["vlim"], 0.04, 0.0025)
        s.treat_reflect()
    return {"r": s.get("r"), "v": s.get("v"), "w": s.get("w"), "F": s.get("F"),
            "nnz": np.array(nnz, dtype=np.int64)}


# -------------------------------------------------------------------- work
def work(case):
    """Bytes: per step every particle's state read once and written once, and
    the snapshot; operations: the pairs within range, each once."""
    kind = case["kind"]
    if kind in ("force", "run", "nlist", "gauss"):
        n, steps = case["n"], case.get("steps", 1)
        pairs = 0.5 * n * case["rho"] * 4.0 / 3.0 * math.pi * RC ** 3
        return {"bytes": n * (98.0 * steps + (24.0 if kind == "force" else 48.0)),
                "flops": 27.0 * pairs * steps}
    if kind in ("batch", "gr"):
        sizes = [s.n for s in _sizes(case)]
        if kind == "gr":
            return {"bytes": 24.0 * sum(sizes) + 8.0 * case["nrep"] * case["bins"],
                    "flops": 15.0 * sum(k * (k - 1) // 2 for k in sizes)}
        n = sum(sizes)
        pairs = 0.5 * n * 0.8 * 4.0 / 3.0 * math.pi * RC ** 3
        return {"bytes": n * (98.0 * case["steps"] + 48.0), "flops": 27.0 * pairs * case["steps"]}
    if kind == "sph":
        n = _dam_count(case)
        nb = 4.0 / 3.0 * math.pi * ((1.7 if case["physics"] == "lucy" else 2.6) ** 3)
        return {"bytes": n * (121.0 * case["steps"] + 72.0),
                "flops": 0.5 * n * nb * 60.0 * case["steps"]}
    n = case["n"]
    contacts = (6.0 if case["bed"] else 0.0) * n
    return {"bytes": n * (156.0 * case["steps"] + 96.0) + 52.0 * contacts * case["steps"],
            "flops": 100.0 * contacts * case["steps"]}


class _Size:
    def __init__(self, n):
        self.n = n


def _sizes(case, seed=5):
    u = workloads.uniform53(seed, 3 * case["nrep"], offset=1 << 40).reshape(-1, 3)
    lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
    return [_Size(int(round(math.exp(lo + x * (hi - lo))))) for x in u[:, 0]]


def _dam_count(case):
    dx, layers = case["dx"], 3
    nx, ny, nz = (int(round(a / dx)) for a in (0.4, 0.4, 0.8))
    wx, wy, wz = (int(round(a / dx)) for a in (1.6, 0.4, 0.8))
    wall = (wx + 2 * layers) * (wy + 2 * layers) * (wz + layers) - wx * wy * wz
    return nx * ny * nz + wall


# ------------------------------------------------------------------- exact
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(x):
    return torch.as_tensor(np.ascontiguousarray(x), dtype=torch.float64, device=_dev())


def _pairs(r, lo, hi, rcut, periodic):
    """All ordered pairs (i, j), i != j, closer than rcut (minimum image when
    periodic), sorted by i: cells of at least rcut, 27 neighbours of each.  A
    box of fewer than 3 cells along an axis takes every pair."""
    dev, n = r.device, r.shape[0]
    ext = hi - lo
    if periodic:
        p = r - ext * torch.floor((r - lo) / ext)
    else:
        p = torch.minimum(torch.maximum(r, lo), hi)
    nb = torch.clamp(torch.floor(ext / rcut), min=1).to(torch.int64).tolist()
    if min(nb) < 3:
        i = torch.arange(n, device=dev)
        I, J = torch.meshgrid(i, i, indexing="ij")
        d = r[I] - r[J]
        if periodic:
            d = d - ext * torch.round(d / ext)
        I, J = I[(d * d).sum(2) < rcut * rcut], J[(d * d).sum(2) < rcut * rcut]
        keep = I != J
        return I[keep], J[keep]
    nbt = torch.tensor(nb, device=dev)
    c3 = torch.minimum((torch.floor((p - lo) / ext * nbt)).to(torch.int64), nbt - 1).clamp(min=0)
    cell = (c3[:, 0] * nb[1] + c3[:, 1]) * nb[2] + c3[:, 2]
    order = torch.argsort(cell, stable=True)
    ncell = nb[0] * nb[1] * nb[2]
    count = torch.bincount(cell, minlength=ncell)
    start = torch.cumsum(count, 0) - count
    width = int(count.max())
    slot = torch.arange(n, device=dev) - start[cell[order]]
    table = torch.full((ncell, width), -1, dtype=torch.int64, device=dev)
    table[cell[order], slot] = order
    used = torch.nonzero(count).flatten()
    found = []
    block = max(1, 30_000_000 // (width * width))
    for a in (-1, 0, 1):
        for b in (-1, 0, 1):
            for c in (-1, 0, 1):
                for u in used.split(block):
                    x = torch.stack([u // (nb[1] * nb[2]) + a, (u // nb[2]) % nb[1] + b,
                                     u % nb[2] + c], 1)
                    if periodic:
                        x = x % nbt
                    else:
                        ok = ((x >= 0) & (x < nbt)).all(1)
                        u, x = u[ok], x[ok]
                    if not u.numel():
                        continue
                    v = (x[:, 0] * nb[1] + x[:, 1]) * nb[2] + x[:, 2]
                    ti, tj = table[u], table[v]
                    r2 = torch.zeros((u.numel(), width, width), dtype=torch.float64, device=dev)
                    for k in range(3):
                        d = r[ti, k][:, :, None] - r[tj, k][:, None, :]
                        if periodic:
                            d = d - ext[k] * torch.round(d / ext[k])
                        r2 += d * d
                    m = ((r2 < rcut * rcut) & (ti >= 0)[:, :, None] & (tj >= 0)[:, None, :]
                         & (ti[:, :, None] != tj[:, None, :]))
                    w = m.nonzero()
                    found.append(torch.stack([ti[w[:, 0], w[:, 1]], tj[w[:, 0], w[:, 2]]]))
    ij = torch.cat(found, 1)
    ij = ij[:, torch.argsort(ij[0], stable=True)]
    return ij[0], ij[1]


def _sum_to(n, i, x):
    return torch.zeros((n,) + x.shape[1:], dtype=torch.float64, device=x.device).index_add_(0, i, x)


class _LJ:
    """FP64 LJ forces, potential energies and virials of one box or several."""

    def __init__(self, boxes, types=1):
        self.sizes = [w.n for w in boxes]
        self.n = sum(self.sizes)
        self.box = torch.repeat_interleave(torch.arange(len(boxes), device=_dev()),
                                           torch.tensor(self.sizes, device=_dev()))
        self.lo = _t(np.stack([w.cell[0::2] for w in boxes]))
        self.ext = _t(np.stack([w.cell[1::2] for w in boxes])) - self.lo
        se = _t(boxes[0].sigma_eps).reshape(types, types, 2)
        self.s2, self.eps = se[:, :, 0] ** 2, se[:, :, 1]
        self.type = torch.as_tensor(np.concatenate([w.type for w in boxes]).astype(np.int64),
                                    device=_dev())
        self.r = torch.cat([_t(w.r) for w in boxes])
        self.v = torch.cat([_t(w.v) for w in boxes])
        self.m = torch.cat([_t(w.m) for w in boxes])[:, None]
        self.skin, self.r0 = 0.5, None

    def per_box(self, x):
        return torch.stack([c.sum() for c in x.split(self.sizes)])

    def force(self, r, energies=True):
        if self.r0 is None or float((r - self.r0).norm(dim=1).max()) > 0.5 * self.skin:
            self.r0, at, found = r.clone(), 0, []
            for k, n in enumerate(self.sizes):
                i, j = _pairs(r[at:at + n], self.lo[k], self.lo[k] + self.ext[k], RC + self.skin,
                              True)
                found.append(torch.stack([i, j]) + at)
                at += n
            self.i, self.j = torch.cat(found, 1)
        i, j = self.i, self.j
        L = self.ext[self.box[i]] if len(self.sizes) > 1 else self.ext[0]
        d = r[i] - r[j]
        d = d - L * torch.round(d / L)
        r2 = (d * d).sum(1)
        near = r2 < RC * RC
        i, j, d, r2 = i[near], j[near], d[near], r2[near]
        ti, tj = self.type[i], self.type[j]
        eps, s6 = self.eps[ti, tj], (self.s2[ti, tj] / r2) ** 3
        c6 = (self.s2[ti, tj] / (RC * RC)) ** 3
        fr = 24.0 * eps * s6 * (2.0 * s6 - 1.0) / r2
        F = _sum_to(self.n, i, fr[:, None] * d)
        if not energies:
            return F, None, None
        pe = 0.5 * _sum_to(self.n, i, 4.0 * eps * (s6 * (s6 - 1.0) - c6 * (c6 - 1.0)))
        return F, self.per_box(pe), self.per_box(0.5 * _sum_to(self.n, i, fr * r2))

    def wrap(self, r):
        lo, L = self.lo[self.box], self.ext[self.box]
        return r - L * torch.floor((r - lo) / L)


def _exact_run(boxes, types, steps, every):
    lj = _LJ(boxes, types)
    r, v, m = lj.r, lj.v, lj.m
    old = torch.zeros_like(r)
    e = []
    for k in range(steps):
        record = bool(every) and k % every == 0
        F, pe, vir = lj.force(r, record)
        v = v + (F + old) * (0.5 * DT / m)
        if record:
            e.append(torch.stack([0.5 * lj.per_box((m * v * v).sum(1)), pe, vir], 1))
        r = r + v * DT + F * (0.5 * DT * DT / m)
        old = F
    return _host(lj.wrap(r)), _host(v), _host(torch.stack(e)) if e else None


def _host(x):
    return x.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "gr":
        return None                       # whole numbers
    if kind == "force":
        lj = _LJ([_fluid(case, seed)], case["types"])
        F, pe, vir = lj.force(lj.r)
        return {"pe": _host(pe), "w": _host(vir), "F": _host(F)}
    if kind == "batch" and case["nrep"] * case["steps"] > 6000:
        return None                       # half a minute and more
    if kind in ("run", "batch", "nlist"):
        boxes = _replicas(case, seed).systems if kind == "batch" else [_fluid(case, seed)]
        r, v, e = _exact_run(boxes, case.get("types", 1), case["steps"],
                             1 if kind == "nlist" else case["every"])
        out = {"r": r, "v": v}
        if kind == "nlist":
            out["pe_w"] = e[:, 0, 1:]
        elif case["every"]:
            out["e"] = e
        return out
    if kind == "gauss":
        return _exact_gauss(case, seed)
    if kind == "sph":
        return _exact_sph(case, seed)
    return _exact_dem(case, seed)


def _exact_gauss(case, seed):
    lj = _LJ([_fluid(case, seed)])
    r, v, m = lj.r, lj.v, lj.m
    old, xi, t = torch.zeros_like(r), 0.0, []
    for _ in range(case["steps"]):
        F, _pe, _w = lj.force(r)
        t.append(float((m * v * v).sum()))
        half = v + (F + old) * (0.5 * DT / m)
        A = half - v * (0.5 * DT * xi)
        # the reference loop's first Newton pass, taken when it moves v by no
        # more than the threshold; else the converged solution
        q = (A - (0.5 * DT * xi + 1.0) * half) / (
            -0.5 * DT * (xi + (F - 2.0 * xi * m * half) * half / (m * half * half).sum()) - 1.0)
        if math.sqrt(float((q * q).sum()) / (3.0 * lj.n)) > 1e-10:
            g = float((F * A).sum() / (m * A * A).sum())
            v = A * (1.0 - 0.5 * DT * g)
            xi = g / (1.0 - 0.5 * DT * g)
        else:
            v = half - q
            xi = float((F * v).sum() / (m * v * v).sum())
        r = r + v * (DT - xi * 0.5 * DT * DT) + F * (0.5 * DT * DT / m)
        old = F
        r = lj.wrap(r)
    return {"r": _host(r), "v": _host(v), "mv2": np.array(t)}


def _exact_sph(case, seed):
    w = _dam(case, seed)
    lo, hi = _t(w.cell[0::2]), _t(w.cell[1::2])
    r, m = _t(w.r), _t(w.m)
    v = torch.zeros_like(r)
    move = _t(1.0 - w.fixed)[:, None]
    lucy = case["physics"] == "lucy"
    h, c0 = w.h, float(w.c[0])
    sup = h if lucy else 2.0 * h
    dt = 0.25 * h / c0
    pad = 2.0 * w.dx
    mu0 = _t(w.mu0)
    i, j = _pairs(r, lo, hi, sup + pad, False)
    moved = 0.0
    num = None
    for _ in range(case["steps"]):
        d = r[i] - r[j]
        R = (d * d).sum(1).sqrt()
        near = R < sup
        I, J, d, R = i[near], j[near], d[near], R[near]
        if lucy:
            w0 = 105.0 / (16.0 * math.pi * h ** 7)
            W = w0 * (h + 3.0 * R) * (h - R) ** 3
            W0 = w0 * h ** 4
            den = _sum_to(w.n, I, torch.stack([W, m[J] * W, mu0[J] * m[J] * W], 1))
            n0, rho, mu = den[:, 0] + W0, den[:, 1] + m * W0, den[:, 2] + mu0 * m * W0
            mu = mu / rho
            num = torch.stack([n0, rho, mu], 1)
            P = c0 * c0 / rho * (1.0 - 1.0 / rho)
            mw = (m[J] * (-12.0 * w0) * (h - R) ** 2)[:, None]
            v1 = ((mu[I] + mu[J]) / (rho[I] * rho[J]))[:, None]
            a = _sum_to(w.n, I, mw * (-d * (P[I] + P[J])[:, None] - (v[J] - v[I]) * v1))
        else:
            ws = 1.0 / (math.pi * h ** 3)
            q = R / h
            W = ws * (0.25 * (2.0 - q) ** 3 - torch.clamp(1.0 - q, min=0.0) ** 3)
            den = _sum_to(w.n, I, torch.stack([W, m[J] * W], 1))
            n0, rho = den[:, 0] + ws, den[:, 1] + m * ws
            p = torch.clamp(w.rho0 * c0 * c0 / 7.0 * ((rho / w.rho0) ** 7 - 1.0), min=0.0)
            num = torch.stack([n0, rho, p], 1)
            g = torch.where(q < 1.0, 2.25 * q - 3.0, -0.75 * (2.0 - q) ** 2 / q) * (ws / h ** 2)
            vr = ((v[I] - v[J]) * d).sum(1)
            visc = torch.where(vr < 0.0, -0.1 * c0 * h * vr /
                               ((R * R + 0.01 * h * h) * 0.5 * (rho[I] + rho[J])), 0.0 * vr)
            P = p / rho ** 2
            a = _sum_to(w.n, I, (-m[J] * (P[I] + P[J] + visc) * g)[:, None] * d)
        a[:, 2] -= 9.81
        v = v + a * dt * move
        r = r + v * dt * move
        r = torch.minimum(torch.maximum(r, lo), hi)
        moved += 2.0 * dt * float(v.norm(dim=1).max())
        if moved > pad:
            i, j = _pairs(r, lo, hi, sup + pad, False)
            moved = 0.0
    return {"r": _host(r), "v": _host(v), "num": _host(num)}


def _exact_dem(case, seed):
    w = _grains(case, seed)
    lo, hi = _t(w.cell[0::2]), _t(w.cell[1::2])
    r, v, m, rad = _t(w.r), _t(w.v), _t(w.m), _t(w.rad)
    dt, n = _dem_dt(case), w.n
    L, om = torch.zeros_like(r), torch.zeros_like(r)
    inertia = (0.4 * rad * rad * m)[:, None]
    pad = 0.2 * float(rad.max())
    # the steps here move a sphere by far less than the margin
    i, j = _pairs(r, lo, hi, 2.0 * float(rad.max()) + pad, False)
    linear = case["law"] == "linear"
    hist = torch.zeros((i.numel(), 3 if linear else 1), dtype=torch.float64, device=r.device)
    F = torch.zeros_like(r)
    for _ in range(case["steps"]):
        d = r[i] - r[j]
        R2 = (d * d).sum(1)
        rs = rad[i] + rad[j]
        hit = R2 < rs * rs
        hist = torch.where(hit[:, None], hist, torch.zeros_like(hist))
        I, J, d, rs = i[hit], j[hit], d[hit], rs[hit]
        R = R2[hit].sqrt()
        nv = d / R[:, None]
        xi = rs - R
        vij = v[I] - v[J]
        vn = (vij * nv).sum(1)
        hh = hist[hit]
        if linear:
            P = DEM_LINEAR
            le = math.log(P["e"])
            zeta = -le / math.sqrt(math.pi ** 2 + le * le)
            meff = 1.0 / (1.0 / m[I] + 1.0 / m[J])
            fn = P["kn"] * xi - 2.0 * zeta * (meff * P["kn"]).sqrt() * vn
            W = rad[I][:, None] * om[I] + rad[J][:, None] * om[J]
            vt = vij - torch.linalg.cross(W, nv) - vn[:, None] * nv
            sp = hh - (hh * nv).sum(1)[:, None] * nv + vt * dt
            ft = -P["kt"] * sp
            size, cap = ft.norm(dim=1), P["mu"] * fn.abs()
            ft = torch.where((size > cap)[:, None], ft * (cap / size)[:, None], ft)
            hh = -ft / P["kt"]
            f = fn[:, None] * nv + ft
            t = -rad[I][:, None] * torch.linalg.cross(nv, ft)
        else:
            P = DEM_HERTZ
            E = P["E"] * (1.0 - P["sigma"] ** 2)
            s2 = (2.0 - P["sigma"]) / 2.0 / (1.0 - P["sigma"])
            mbar = 1.0 / (1.0 / m[I] + 1.0 / m[J])
            Kn = 2.0 / 3.0 * E * (rad[I] * rad[J] / rs * xi).sqrt()
            Fn = nv * (Kn * xi - P["gamma"] * (mbar * Kn).sqrt() * vn)[:, None]
            F0 = Fn.norm(dim=1)
            arm = (-rad[I] / rs)[:, None] * d
            vt = vij - vn[:, None] * nv + torch.linalg.cross(om[I] + om[J], arm)
            slip = (vt != 0).all(1)
            size = torch.where(slip, vt.norm(dim=1), torch.ones_like(F0))
            xsm = P["mu"] * s2 * xi
            part = torch.where(hh[:, 0] < xsm, hh[:, 0] / xsm, torch.ones_like(xsm))
            Fs = torch.where(slip[:, None], (-P["mu"] * F0 * part / size)[:, None] * vt, 0.0 * vt)
            hh = hh + torch.where(slip, size * dt, 0.0 * size)[:, None]
            spin = (om[I] != 0).all(1)
            wn = torch.where(spin, om[I].norm(dim=1), torch.ones_like(F0))
            Tr = torch.where(spin[:, None], (-P["mu_r"] * rad[I] * F0 / wn)[:, None] * om[I],
                             0.0 * vt)
            f = Fn + Fs
            t = torch.linalg.cross(arm, Fs) + Tr
        hist[hit] = hh
        F, T = _sum_to(n, I, f), _sum_to(n, I, t)
        a = F / m[:, None]
        a[:, 2] -= 9.8
        v = v + a * dt
        r = r + v * dt
        L = L + T * dt
        om = L / inertia
        v = torch.where(r < lo, v.abs(), torch.where(r > hi, -v.abs(), v))
    return {"r": _host(r), "v": _host(v), "w": _host(om), "F": _host(F), "nnz": None}
