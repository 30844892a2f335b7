"""The workloads by which this engine's speed is judged.

Each case is what a user's molecular-dynamics, sampling or fitting program
has the engine do, through the Python binding of the C ABI: single force
calls on host arrays (the drop-in path), device-resident RESPA runs in the
NVE, NVT and NPT ensembles, batched HMC chains, fluid in a tube on a
tabulated wall, and parameter gradients for force-field fitting.  Models and
settings are those of mspms2_amd.configs and bench.py.  Starting structures
are made here from the seed alone (water: a hydrogen-bonded cubic-ice
lattice at the density of the 12,288-site box, displaced and turned at
random), so that every run of a case starts from the same numbers.

`exact` restates each path in plain torch in 64 bits: pair sums over a list
of all pairs within the cutoff, the Ewald sum by complex matrix products,
bonded forces by autograd, the integrators step by step.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from mspms2_amd import abi, configs, sfgrid
from mspms2_amd.autograd import NonbondedEnergy, site_params
from mspms2_amd.engine import LONG_TERMS_BYTES, SHORT_TERMS_BYTES, Engine
from mspms2_amd.runio import RunDir, RunInput
from mspms2_amd.system import System

LT, ST = LONG_TERMS_BYTES // 8, SHORT_TERMS_BYTES // 8
NLT = len(abi.LongTerms.ENERGY_FIELDS)     # the energies; pair counts follow them

CELL = (8.0 * 49.66 ** 3 / 4096.0) ** (1.0 / 3.0)   # 8 waters per cubic cell


# ---- the cases -------------------------------------------------------------
def listed():
    return [
        # one drop-in frclong + frcshort call on host arrays: a small box, as a
        # host-driven integrator or a Monte Carlo program makes them (latency)
        dict(name="call_water_216_mixed", kind="call", mols=216, precision="mixed"),
        # the same calls on the 12,288-site box in the exact mode, the drop-in's
        # reference-order setting
        dict(name="call_water_4096_fp64", kind="call", mols=4096, precision="fp64"),
        # a small NVE box: every kernel is short, launches and gaps count
        dict(name="nve_water_216_mixed", kind="nve", mols=216, precision="mixed", steps=24),
        # the headline workload: 12,288 sites, every step's terms recorded
        dict(name="nve_water_4096_mixed", kind="nve", mols=4096, precision="mixed", steps=20),
        # an odd count with vacancies in the exact mode
        dict(name="nve_water_1003_fp64", kind="nve", mols=1003, precision="fp64", steps=10),
        # the largest Ewald box the k tables take at this accuracy (kmax 16)
        dict(name="nve_water_32768_mixed", kind="nve", mols=32768, precision="mixed", steps=4),
        # the reference's argon run: LJ-864, Nose-Hoover NVT
        dict(name="nvt_argon_864_mixed", kind="nvt_argon", cells=6, precision="mixed", steps=40),
        # Nose-Hoover RESPA of the headline box
        dict(name="nvt_water_4096_mixed", kind="nvt", mols=4096, precision="mixed", steps=6),
        # constant pressure, an odd count, the exact mode
        dict(name="npt_water_999_fp64", kind="npt", mols=999, precision="fp64", steps=6),
        # sampling: one HMC move (10 RESPA steps) of 64 butane boxes of 64-512
        # molecules, one chain per box
        dict(name="hmc_butane_64", kind="hmc", boxes=64, lo=64, hi=512, precision="mixed"),
        # adsorption: two methane loadings in a 50 A tube, the wall a 512 MiB
        # Hermite grid evaluated in the inner loop
        dict(name="tube_2x40000", kind="tube", boxes=2, sites=40000, steps=16),
        # force-field fitting: energies, forces and parameter gradients of 16
        # Wolf-water configurations, forward and backward
        dict(name="fit_wolf_16x1024", kind="fit", boxes=16, mols=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["call", "call", "nve", "nve", "nve", "nvt_argon", "nvt", "npt", "hmc",
                       "tube", "fit"])
    if kind == "call":
        return dict(kind=kind, mols=_log(rng, 150, 5000), precision=rng.choice(["mixed", "fp64"]))
    if kind == "nve":
        prec = rng.choice(["mixed", "mixed", "fp64"])
        n = _log(rng, 150, 30000 if prec == "mixed" else 4500)
        return dict(kind=kind, mols=n, precision=prec, steps=20 if n < 6000 else 4)
    if kind == "nvt_argon":
        return dict(kind=kind, cells=rng.randint(4, 20), precision=rng.choice(["mixed", "fp64"]),
                    steps=20)
    if kind == "nvt":
        return dict(kind=kind, mols=_log(rng, 200, 6000), precision=rng.choice(["mixed", "fp64"]),
                    steps=6)
    if kind == "npt":
        return dict(kind=kind, mols=_log(rng, 400, 3000), precision=rng.choice(["mixed", "fp64"]),
                    steps=5)
    if kind == "hmc":
        return dict(kind=kind, boxes=rng.randint(3, 80), lo=64, hi=rng.randint(100, 512),
                    precision="mixed")
    if kind == "tube":
        return dict(kind=kind, boxes=rng.randint(1, 3), sites=_log(rng, 10000, 40000), steps=16)
    return dict(kind="fit", boxes=rng.randint(2, 20), mols=rng.randint(520, 1024))


# ---- systems ---------------------------------------------------------------
def _cells_for(nmol):
    """The near-cubic (nx, ny, nz) of 8-molecule cells that holds nmol with
    the fewest vacancies."""
    c = max(3, round((nmol / 8.0) ** (1.0 / 3.0)))
    best = None
    for x in range(max(3, c - 1), c + 2):
        for y in range(x, x + 3):
            for z in range(y, x + 3):
                if 8 * x * y * z >= nmol and (best is None or x * y * z < best[0]):
                    best = (x * y * z, (x, y, z))
    return best[1]


@functools.lru_cache(maxsize=4)
def _ice(nx, ny, nz):
    """Proton-ordered cubic ice: oxygens on the diamond lattice, each water's
    two protons towards its two neighbours above it along z, so that each
    O..O contact holds one proton.  (8 nx ny nz, 3 sites, 3)."""
    fcc = np.array([[0, 0, 0], [0, .5, .5], [.5, 0, .5], [.5, .5, 0]])
    dirs = {0: [(1, 1, 1), (-1, -1, 1)], 1: [(-1, 1, 1), (1, -1, 1)]}
    tmpl = np.array([[s.xx, s.yy, s.zz] for s in configs.water_species(1).sites])
    basis = []
    for sub in (0, 1):
        h = np.array(dirs[sub], dtype=np.float64) / math.sqrt(3.0)
        axis, flat = h.sum(0), h[0] - h[1]
        axis, flat = axis / np.linalg.norm(axis), flat / np.linalg.norm(flat)
        mol = tmpl[:, :1] * flat + tmpl[:, 2:] * axis
        for f in fcc + 0.25 * sub + 0.125:
            basis.append(f * CELL + mol)
    g = np.stack(np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij"), -1)
    return (g.reshape(-1, 1, 1, 1, 3) * CELL + np.array(basis)[None]).reshape(-1, 3, 3)


def _turned(rng, n, most):
    """Rotation matrices about random axes by angles of up to `most`."""
    u = rng.standard_normal((n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    t = most * rng.random(n)
    K = np.zeros((n, 3, 3))
    K[:, 0, 1], K[:, 0, 2], K[:, 1, 2] = -u[:, 2], u[:, 1], -u[:, 0]
    K -= K.transpose(0, 2, 1)
    return np.eye(3) + np.sin(t)[:, None, None] * K + (1 - np.cos(t))[:, None, None] * (K @ K)


def _water(nmol, seed, elec="ewald", rc=10.0, kappa=0.28, ensemble=0):
    rng = np.random.default_rng(seed)
    cells = _cells_for(nmol)
    xyz = _ice(*cells)
    xyz = xyz[np.sort(rng.permutation(len(xyz))[:nmol])]
    # molecules turned by up to 0.25 rad and moved by up to 0.12 A per axis,
    # bond lengths off by up to 0.02 A
    o = xyz[:, :1]
    xyz = o + np.einsum("nsk,njk->nsj", xyz - o, _turned(rng, nmol, 0.25))
    xyz = xyz + rng.uniform(-0.12, 0.12, (nmol, 1, 3)) + rng.uniform(-0.02, 0.02, xyz.shape)
    L = [c * CELL for c in cells]
    rc = min(rc, 0.49 * min(L))
    k = [max(3, min(16, round(8 * v / 49.66))) for v in L]
    run = RunInput(title=f"water {nmol}", treq=298.0, preq=1.0, boxlx=L[0], boxly=L[1],
                   boxlz=L[2], rcuton=rc, rcutoff=rc, rcutoffelec=rc, delt=2.0, nstep_inner=8,
                   what_ensemble=ensemble,
                   iChargeType=abi.ELEC_EWALD if elec == "ewald" else abi.ELEC_WOLF, kappa=kappa,
                   kmaxx=k[0], kmaxy=k[1], kmaxz=k[2], ksqmax=max(k) ** 2,
                   fEwald_BC=abi.EWALD_BC_TINFOIL, fEwald_Dim=3)
    return System.from_rundir(RunDir(run=run, sysname="water",
                                     species=[configs.water_species(nmol)],
                                     xyz=np.ascontiguousarray(xyz.reshape(-1, 3))))


def _butane(nmol, seed):
    """configs.butane_box's box and columns, all chains placed at once."""
    rng = np.random.default_rng(seed)
    L = (nmol / configs.BUTANE_DENSITY) ** (1.0 / 3.0)
    nz = max(1, int(L / 6.9))
    nxy = int(math.ceil(math.sqrt(nmol / nz)))
    sites = np.stack(np.meshgrid(np.arange(nxy), np.arange(nxy), np.arange(nz), indexing="ij"),
                     -1).reshape(-1, 3)
    at = (sites[np.sort(rng.permutation(len(sites))[:nmol])] + 0.5) * \
        np.array([L / nxy, L / nxy, L / nz])
    t = configs.BUTANE_TMPL - configs.BUTANE_TMPL.mean(0)
    _, V = np.linalg.eigh(t.T @ t)
    t = t @ V[:, ::-1][:, [1, 2, 0]]
    s = 2 * np.pi * rng.random(nmol)
    spin = np.zeros((nmol, 3, 3))
    spin[:, 0, 0] = spin[:, 1, 1] = np.cos(s)
    spin[:, 1, 0], spin[:, 0, 1] = np.sin(s), -np.sin(s)
    spin[:, 2, 2] = 1.0
    rot = _turned(rng, nmol, 0.1) @ spin
    xyz = at[:, None] + np.einsum("sk,njk->nsj", t, rot) + rng.uniform(-0.1, 0.1, (nmol, 1, 3))
    rc = min(14.0, 0.5 * L * (1 - 1e-12))
    run = RunInput(title=f"n-butane {nmol}", treq=300.0, boxlx=L, boxly=L, boxlz=L, rcuton=rc,
                   rcutoff=rc, rcutoffelec=rc, delt=1.0, nstep_inner=5, what_simulation=1,
                   iChargeType=abi.ELEC_NONE, nstep_md_per_hmc=10)
    return System.from_rundir(RunDir(run=run, sysname="n-butane",
                                     species=[configs.butane_species(nmol)],
                                     xyz=np.ascontiguousarray(xyz.reshape(-1, 3))))


@functools.lru_cache(maxsize=1)
def _tube_wall():
    """The 128 x 128 x 1024 grid file of the 50 A tube (no seed: a table that
    a user has on disk)."""
    h = 100.0 / 127.0
    return sfgrid.tube_grid([(3.73, 148.0)], R=50.0, x0=-50.0, y0=-50.0, nx=128, ny=128, hx=h,
                            hy=h, nz=1024, hz=4000.0 / 1023.0, sigma_s=3.37, eps_s=27.68)


def _systems(case, seed):
    k = case["kind"]
    if k in ("call", "nve", "nvt", "npt"):
        return [_water(case["mols"], seed, rc=9.0 if k == "npt" else 10.0,
                       ensemble={"nvt": 1, "npt": 2}.get(k, 0))]
    if k == "nvt_argon":
        return [System.from_rundir(configs.lj_fcc(ncell=case["cells"], jitter=0.05, seed=seed))]
    if k == "hmc":
        # the box sizes are the workload's, not the seed's
        n = np.random.default_rng(2024).integers(case["lo"], case["hi"] + 1, size=case["boxes"])
        return [_butane(int(v), 1000 * (seed % 100000) + r) for r, v in enumerate(n)]
    if k == "tube":
        out = [System.from_rundir(configs.tube_loading(case["sites"] + 1001 * r,
                                                       seed=100 * (seed % 100000) + r))
               for r in range(case["boxes"])]
        for s in out:
            s.grid = _tube_wall()
        return out
    return [_water(case["mols"], 1000 * (seed % 100000) + r, elec="wolf", rc=12.0, kappa=0.2)
            for r in range(case["boxes"])]


def _velocities(s, seed, temp):
    """Maxwell-Boltzmann velocities at `temp` (reduced), no total momentum."""
    rng = np.random.default_rng(seed + 77)
    m = s.masses()
    v = rng.standard_normal((3, s.natom)) * np.sqrt(temp / m)
    return v - (v * m).sum(axis=1, keepdims=True) / m.sum()


def _xyz(s):
    return np.stack([s.xx, s.yy, s.zz])


def _start_velocities(case, systems, seed):
    # the ice starts at twice the run's temperature: half of the kinetic
    # energy goes into the lattice, which melts
    hot = 2.0 if case["kind"] == "nve" else 1.0
    return np.concatenate([_velocities(s, seed + r, hot * s.treq)
                           for r, s in enumerate(systems)], axis=1)


def _moved(s, seed):
    """Two position sets of the host calls: the second after a small move."""
    rng = np.random.default_rng(seed + 5)
    x = _xyz(s)
    return [x, x + rng.uniform(-0.01, 0.01, x.shape)]


def _params(systems):
    """Two parameter sets of a fit, as an optimiser's steps leave them."""
    p = site_params(systems[0])
    return [tuple(v.clone() for v in p), tuple(v * (1.0 + 1e-3 * (i + 1)) for i, v in enumerate(p))]


# ---- what a program keeps, and one pass -------------------------------------
@functools.lru_cache(maxsize=1)
def _stream():
    """The stream of the program's device runs, one for all its engines."""
    return torch.cuda.Stream()


def prepare(case, seed):
    kind = case["kind"]
    systems = _systems(case, seed)
    s = systems[0]
    if kind == "call":
        return dict(kind=kind, eng=Engine(s, precision=case["precision"]), x=_moved(s, seed), k=0)
    if kind == "fit":
        eng = Engine.replicas(systems, precision="fp64")
        return dict(kind=kind, eng=eng, k=0, params=_params(systems),
                    pos=torch.tensor(eng.packed_positions()),
                    target=torch.tensor(-20000.0 * case["mols"], dtype=torch.float64))
    dev = torch.device("cuda:0")
    if len(systems) > 1 or kind in ("hmc", "tube"):
        eng = Engine.replicas(systems, precision=case.get("precision", "mixed"))
        x = eng.packed_positions()
    else:
        eng, x = Engine(s, precision=case["precision"]), _xyz(s)
    nr, K = len(systems), case.get("steps", 1)
    new = lambda n: torch.zeros(n, dtype=torch.float64, device=dev)  # noqa: E731
    st = dict(kind=kind, eng=eng, pos=torch.tensor(x, device=dev), lt=new(nr * LT),
              sterms=new(nr * ST), uk=new(nr), steps=K, nrep=nr, delt=s.delt,
              inner=s.run.nstep_inner, lh=new(K * nr * LT), sh=new(K * nr * ST), kh=new(K * nr))
    v = _start_velocities(case, systems, seed)
    nfree = 3 * s.natom - s.run.nconstraint
    if kind == "nve":
        eng.set_list_skin(5.0 if case["precision"] == "mixed" and s.natom > 6000 else 2.5)
    elif kind == "nvt_argon":
        q = 100.0 * s.natom / 864.0
        eng.nvt_set(q, q, s.treq, nfree)
        eng.set_list_skin(0.3)
    elif kind == "nvt":
        eng.nvt_set(4.0 * nfree, 4.0 * nfree, s.treq, nfree)
        eng.set_list_skin(5.0 if case["precision"] == "mixed" and s.natom > 6000 else 2.5)
    elif kind == "npt":
        eng.npt_set(4.0 * nfree, 400.0 * nfree, s.treq, s.preq, nfree, vts=0.0, vbs=0.0)
    elif kind == "tube":
        eng.set_sf_split(True)
        eng.set_list_skin(1.0)
    if kind == "hmc":
        st["vel"], st["fl"], st["fs"] = (torch.zeros_like(st["pos"]) for _ in range(3))
        eng.hmc_init([1000 + r + seed % 20000 for r in range(nr)], [2000 + r for r in range(nr)],
                     [q.treq for q in systems], [q.run.nconstraint for q in systems], st["vel"])
        return st
    st["vel"] = torch.tensor(v, device=dev)
    # the starting forces, and the terms that the barostat reads
    st["fl"], st["fs"] = torch.zeros_like(st["pos"]), torch.zeros_like(st["pos"])
    fl, _ = eng.frclong(*x)
    st["fl"].copy_(torch.tensor(fl))
    eng.frcshort_device(st["pos"], st["fs"], st["sterms"])
    if kind == "npt":
        eng.frclong_device(st["pos"], st["fl"], st["lt"])
    eng.sync()
    if kind == "tube":
        # a study of one loading starts its runs from a stored configuration
        st["start"] = [st[k].clone() for k in ("pos", "vel", "fl", "fs")]
    return st


def run(st):
    kind, eng = st["kind"], st["eng"]
    if kind == "call":
        x = st["x"][st["k"] % 2]
        st["k"] += 1
        fl, tl = eng.frclong(x[0], x[1], x[2])
        fs, ts = eng.frcshort(x[0], x[1], x[2])
        return dict(fl=fl, fs=fs, long=np.array([tl[k] for k in abi.LongTerms.ENERGY_FIELDS]),
                    short=np.array([ts[k] for k in _SHORT]))
    if kind == "fit":
        eps, sig, q = (v.requires_grad_() for v in st["params"][st["k"] % 2])
        st["k"] += 1
        pos = st["pos"].requires_grad_()
        e = NonbondedEnergy.apply(pos, eps, sig, q, eng)
        loss = ((e - st["target"]) / 1e6).square().mean()
        g = torch.autograd.grad(loss, (pos, eps, sig, q))
        return dict(energy=e.detach(), loss=loss.detach(), dpos=g[0], deps=g[1], dsig=g[2],
                    dq=g[3])
    pos, vel, fl, fs = st["pos"], st["vel"], st["fl"], st["fs"]
    lt, sm, uk, d, nin, K, nr = (st["lt"], st["sterms"], st["uk"], st["delt"], st["inner"],
                                 st["steps"], st["nrep"])
    out = dict(pos=pos, vel=vel, fl=fl, fs=fs, long=lt.view(nr, LT)[:, :NLT],
               short=sm.view(nr, ST), ukin=uk)
    on = dict(graph=True, stream=_stream().cuda_stream)
    if kind in ("nve", "tube"):
        if "start" in st:
            with torch.cuda.stream(_stream()):
                for k, v in zip(("pos", "vel", "fl", "fs"), st["start"]):
                    st[k].copy_(v)
        eng.vver_run_device(pos, vel, fl, fs, d, nin, K, lt, sm, uk, lhist=st["lh"],
                            shist=st["sh"], ukin_hist=st["kh"], **on)
        out.update(lhist=st["lh"].view(K, nr, LT)[:, :, :NLT], shist=st["sh"].view(K, nr, ST),
                   khist=st["kh"])
    elif kind in ("nvt", "nvt_argon"):
        eng.nvt_run_device(pos, vel, fl, fs, d, nin, K, lt, sm, uk, **on)
    elif kind == "npt":
        eng.npt_run_device(pos, vel, fl, fs, d, nin, K, lt, sm, uk, **on)
    else:
        eng.hmc_run_device(pos, vel, fl, fs, d, nin, 10, 1, lt, sm, uk, **on)
    return out


_SHORT = [n for n, _ in abi.ShortTerms._fields_]


# ---- the work it cannot do without -------------------------------------------
def _pairs(natom, vol, rc):
    return 0.5 * natom * natom / vol * 4.0 / 3.0 * math.pi * rc ** 3


def work(case):
    """Bytes: every input read and every output written once per pass (a run
    of K steps keeps its state on the chip's side: positions, velocities and
    both forces in and out once).  Operations: per force evaluation 20 per
    pair for the geometry, 24 for LJ, 25 for Ewald or Wolf, 12 per half-space
    k vector and site (structure factor and force as matrix products), 60
    per bond, 90 per angle, 250 per dihedral and inner step, 1064 per grid
    lookup; the parameter gradients about double a pair's work."""
    k, K = case["kind"], case.get("steps", 1)
    if k in ("call", "nve", "nvt", "npt"):
        cells = _cells_for(case["mols"])
        L = [c * CELL for c in cells]
        n, vol = 3 * case["mols"], L[0] * L[1] * L[2]
        rc = min(9.0 if k == "npt" else 10.0, 0.49 * min(L))
        p = _pairs(n, vol, rc)
        km = [max(3, min(16, round(8 * v / 49.66))) for v in L]
        g = np.meshgrid(*(np.arange(-v, v + 1) for v in km), indexing="ij")
        nk = (int((sum(v * v for v in g) <= max(km) ** 2).sum()) - 1) / 2
        inner = 8 if k != "call" else 1
        flops = K * (p * 45 + p / 9 * 24 + 12.0 * nk * n + inner * case["mols"] * 210)
        return dict(bytes=8.0 * n * (9 if k == "call" else 24), flops=flops)
    if k == "nvt_argon":
        n = 4 * case["cells"] ** 3
        return dict(bytes=8.0 * n * 24, flops=K * (_pairs(n, n / 0.8442, 2.5) * 44 + 60.0 * n))
    if k == "hmc":
        m = case["boxes"] * (case["lo"] + case["hi"]) / 2
        n = 4 * m
        p = _pairs(n, n / (4 * configs.BUTANE_DENSITY), 14.0)
        return dict(bytes=8.0 * n * 24, flops=11 * p * 44 + 50 * m * (180 + 180 + 250))
    if k == "tube":
        n = sum(case["sites"] + 1001 * r for r in range(case["boxes"]))
        p = case["boxes"] * _pairs(n / case["boxes"], math.pi * 46.0 ** 2 * 4000.0, 12.0)
        # the grid's cells inside the tube are read at most once each
        grid = min(256.0 * n, math.pi / 4 * 128 * 128 * 1024 * 32.0)
        return dict(bytes=8.0 * n * 24 + grid, flops=K * (p * 44 + 4 * 1064.0 * n))
    n = 3 * case["mols"]
    p = _pairs(n, case["mols"] / 8 * CELL ** 3, 12.0) * case["boxes"]
    return dict(bytes=8.0 * n * case["boxes"] * 9, flops=p * 2 * 45 + p / 9 * 2 * 24)


def tolerance(case):
    """About four times what a run's error against `exact` was measured at, a
    trajectory's after the few passes that are compared."""
    k = case["kind"]
    if k == "fit" or case.get("precision") == "fp64":
        # sums of 64-bit terms in another order (measured 1e-13 to 4e-12)
        return dict(rel=1e-10, max=1e-8)
    if k == "call":
        return dict(rel=6e-6, max=2e-4)     # 32-bit pair terms (1.2e-6)
    return dict(rel=3e-5, max=1e-3)         # and a trajectory of them (2.4e-6 in one pass)


# ---- the same in 64 bits, in plain torch --------------------------------------
def _t(a):
    dev = "cuda:0" if torch.cuda.is_available() else "cpu"
    return torch.as_tensor(np.array(a), dtype=torch.float64, device=dev)


class _Exact:
    """frclong / frcshort of one system of three-site waters or single LJ
    sites: forces and the terms, on (3, N) positions."""

    def __init__(self, s):
        p = s.params
        self.s, self.n, self.nm, self.per = s, s.natom, s.species[0].nmole, s.species[0].natom
        self.L = _t([p["boxlx"], p["boxly"], p["boxlz"]])
        self.rc = p["rcutoff"]
        self.q, self.m = _t(s.charges()), _t(s.masses())
        sp = s.species[0]
        self.sig, self.eps = _t(np.tile(sp.sigma, self.nm)), _t(np.tile(sp.epsilon, self.nm))
        self.lj = _t(np.tile(sp.ghost_type, self.nm)) == 0
        self.elec = p["iChargeType"]
        self.kappa, self.grid = p["kappa"], s.grid
        self.kmax, self.ksq = (p["kmaxx"], p["kmaxy"], p["kmaxz"]), p["ksqmax"]
        # 1 / (4 kappa^2) and the other constants of init_vars; COULOMB 167100.8084
        self.C = 167100.80840 / p["epsilon_base"] / p["sigma_base"]
        self.split = False
        self.b2 = (3 * torch.arange(self.nm, device=self.L.device)) if self.per == 3 else None

    def pairs(self, x):
        """i < j of different molecules within the cutoff, by slabs along z."""
        L, n = self.L, self.n
        ns = int(float(L[2]) / self.rc)
        slab = torch.remainder(x[2] / L[2], 1.0).mul(ns).long().clamp(max=ns - 1)
        order = torch.argsort(slab)
        start = [0] + torch.cumsum(torch.bincount(slab, minlength=ns), 0).tolist()
        mol = torch.arange(n, device=x.device) // self.per
        got = []
        blocks = [(a, b) for a in range(ns) for b in {a, (a + 1) % ns}] if ns > 2 else None
        for a, b in blocks or [(None, None)]:
            i = order[start[a]:start[a + 1]] if blocks else torch.arange(n, device=x.device)
            j = order[start[b]:start[b + 1]] if blocks else i
            step = max(1, 20_000_000 // max(1, len(j)))
            for c in range(0, len(i), step):
                ii = i[c:c + step]
                r2 = torch.zeros(len(ii), len(j), dtype=x.dtype, device=x.device)
                for d in range(3):
                    t = x[d][ii][:, None] - x[d][j][None, :]
                    t -= L[d] * torch.round(t / L[d])
                    r2 += t * t
                ok = (r2 < self.rc * self.rc) & (mol[ii][:, None] != mol[j][None, :])
                if a == b:
                    ok &= ii[:, None] < j[None, :]
                u, v = torch.nonzero(ok, as_tuple=True)
                got.append(torch.stack([ii[u], j[v]]))
        return torch.cat(got, dim=1)

    def _real(self, r, qq):
        """Ewald or Wolf real-space (energy, -dU/dr / r) of charge products."""
        k, rc = self.kappa, self.rc
        spi = math.sqrt(math.pi)
        if self.elec == abi.ELEC_EWALD:
            u = qq * torch.erfc(k * r) / r
            return u, (u + qq * 2 * k / spi * torch.exp(-(k * r) ** 2)) / (r * r)
        e = math.erfc(k * rc)
        v2 = e / rc ** 2 + 2 * k * math.exp(-(k * rc) ** 2) / (spi * rc)
        u = qq * (torch.erfc(k * r) / r - e / rc + v2 * (r - rc))
        f = qq / r * (torch.erfc(k * r) / (r * r) + 2 * k / spi * torch.exp(-(k * r) ** 2) / r
                      - v2)
        return u, f

    def long(self, x):
        L, f = self.L, torch.zeros_like(x)
        i, j = self.pairs(x)
        d = x[:, i] - x[:, j]
        d = d - L[:, None] * torch.round(d / L[:, None])
        r2 = (d * d).sum(0)
        both = self.lj[i] & self.lj[j]
        il, jl, rl = i[both], j[both], r2[both]
        sg, ep = 0.5 * (self.sig[il] + self.sig[jl]), torch.sqrt(self.eps[il] * self.eps[jl])
        s6 = (sg * sg / rl) ** 3
        uvdw = (4 * ep * (s6 * s6 - s6)).sum()
        g = 24 * ep * (2 * s6 * s6 - s6) / rl
        vir = (g * rl).sum()
        sh1 = self.rc ** -6.0
        ushift = 4 * sh1 * (ep * sg ** 6 * (sg ** 6 * sh1 - 1.0)).sum()
        w = torch.zeros_like(r2)
        w[both] = g
        ureal = uexcl = uself = ufour = x.new_zeros(())
        if self.elec:
            u, g = self._real(torch.sqrt(r2), self.C * self.q[i] * self.q[j])
            ureal = u.sum()
            w = w + g
        f.index_add_(1, i, w * d)
        f.index_add_(1, j, -w * d)
        if self.elec:
            for a, b in ((0, 1), (0, 2), (1, 2)):
                ia, ib = self.b2 + a, self.b2 + b
                e = x[:, ia] - x[:, ib]
                r = torch.sqrt((e * e).sum(0))
                qq = self.C * self.q[ia] * self.q[ib]
                u, g = self._real(r, qq)
                ureal, uexcl = ureal + u.sum(), uexcl + (qq / r).sum()
                t = (g - qq / r ** 3) * e
                f[:, ia] += t
                f[:, ib] -= t
            uself = self.C * (self.q * self.q).sum() * self.kappa / math.sqrt(math.pi)
            ufour = self._recip(x, f)
        uelec = ureal + ufour - uself - uexcl
        usf = x.new_zeros(())
        if self.grid is not None:
            usf, fw = self.wall(x)
            if not self.split:
                f += fw
        zero = x.new_zeros(())
        return f, torch.stack([uvdw, ushift, ureal, uexcl, ufour, uself, zero, uelec, usf, zero,
                               uvdw + uelec + usf, vir + uelec])

    def _recip(self, x, f):
        """The half-space Ewald sum by kx plane; adds its forces to f."""
        tl = [2 * math.pi / v for v in self.L.tolist()]
        vf = 2 * math.pi / math.prod(self.L.tolist())
        km = self.kmax
        e = [torch.exp(1j * tl[d] * x[d][:, None] *
                       torch.arange(-km[d], km[d] + 1, device=x.device)) for d in range(3)]
        ky = torch.arange(-km[1], km[1] + 1, device=x.device).to(x.dtype)[:, None]
        kz = torch.arange(-km[2], km[2] + 1, device=x.device).to(x.dtype)[None, :]
        energy, g = x.new_zeros(()), torch.zeros_like(x)
        for kx in range(km[0] + 1):
            k2 = kx * kx + ky * ky + kz * kz
            ok = (k2 <= self.ksq) & (k2 > 0)
            if kx == 0:
                ok &= (ky > 0) | ((ky == 0) & (kz > 0))
            rk = (tl[0] * kx) ** 2 + (tl[1] * ky) ** 2 + (tl[2] * kz) ** 2
            wk = torch.where(ok, 2 * torch.exp(-rk / (4 * self.kappa ** 2)) /
                             torch.where(ok, rk, 1.0), 0.0)
            exy = e[0][:, kx + km[0]][:, None] * e[1]
            S = (self.q[:, None] * exy).T @ e[2]
            energy = energy + (wk * (S * S.conj()).real).sum()
            A = 2 * vf * self.C * wk * S.conj()
            T = e[2] @ A.T                       # sum over kz, (n, ky)
            h = (exy * T).imag
            g[0] += h.sum(1) * (tl[0] * kx)
            g[1] += (h * ky[:, 0]).sum(1) * tl[1]
            g[2] += ((exy * (e[2] @ (A * kz).T)).imag).sum(1) * tl[2]
        f += self.q * g
        return energy * vf * self.C

    def wall(self, x):
        """The tricubic Hermite lookup of every site: energy and forces."""
        G = self.grid
        h = [G["hx"], G["hy"], G["hz"]]
        p = [x[0] - G["x0"], x[1] - G["y0"], x[2] - G["z0"]]
        pz = (G["nz"] - 1) * G["hz"]
        p[2] = p[2] - torch.floor(p[2] / pz) * pz
        idx = [torch.floor(p[d] / h[d]).long() for d in range(3)]
        b, db = [], []
        for d in range(3):
            t = p[d] / h[d] - idx[d]
            b.append([2 * t ** 3 - 3 * t ** 2 + 1, 3 * t ** 2 - 2 * t ** 3,
                      h[d] * (t ** 3 - 2 * t ** 2 + t), h[d] * (t ** 3 - t ** 2)])
            db.append([(6 * t * t - 6 * t) / h[d], (6 * t - 6 * t * t) / h[d],
                       3 * t * t - 4 * t + 1, 3 * t * t - 2 * t])
        nodes = self._nodes()
        field = {(0, 0, 0): 0, (1, 0, 0): 1, (0, 1, 0): 2, (0, 0, 1): 3, (1, 1, 0): 4,
                 (1, 0, 1): 5, (0, 1, 1): 6, (1, 1, 1): 7}
        v, g = torch.zeros_like(x[0]), [torch.zeros_like(x[0]) for _ in range(3)]
        for c in range(8):
            cx, cy, cz = c & 1, (c >> 1) & 1, (c >> 2) & 1
            at = ((idx[2] + cz) * G["ny"] + idx[1] + cy) * G["nx"] + idx[0] + cx
            for (ox, oy, oz), k in field.items():
                w = nodes[k][at].double()
                X, Y, Z = cx + 2 * ox, cy + 2 * oy, cz + 2 * oz
                v += w * b[0][X] * b[1][Y] * b[2][Z]
                g[0] += w * db[0][X] * b[1][Y] * b[2][Z]
                g[1] += w * b[0][X] * db[1][Y] * b[2][Z]
                g[2] += w * b[0][X] * b[1][Y] * db[2][Z]
        v = torch.where(v < 1.5 * self._lowest, -v, v)
        return v.sum(), -torch.stack(g)

    def _nodes(self):
        if not hasattr(self, "_node_table"):
            t = torch.as_tensor(self.grid["nodes"][0], device=self.L.device)
            self._node_table, self._lowest = t.reshape(8, -1), float(t[0].min())
        return self._node_table

    def short(self, x):
        """Bonds and angles (reduced template parameters)."""
        z = x.new_zeros(())
        fs, ub, ua, vir = torch.zeros_like(x), z, z, z
        sp = self.s.species[0]
        if len(sp.bnd_type):
            y = x.detach().requires_grad_()
            with torch.enable_grad():
                ub = ua = 0.0
                for (a, b), (kb, r0, _) in zip(sp.bnd_idx, sp.bnd_para):
                    e = y[:, self.b2 + int(a)] - y[:, self.b2 + int(b)]
                    r = torch.sqrt((e * e).sum(0))
                    ub = ub + (0.5 * kb * (r - r0) ** 2).sum()
                    vir = vir - (kb * (r - r0) * r).detach().sum()
                for (a, b, c), (kt, t0, *_) in zip(sp.agl_idx, sp.agl_para):
                    u = y[:, self.b2 + int(a)] - y[:, self.b2 + int(b)]
                    w = y[:, self.b2 + int(c)] - y[:, self.b2 + int(b)]
                    ct = (u * w).sum(0) / torch.sqrt((u * u).sum(0) * (w * w).sum(0))
                    ua = ua + (0.5 * kt * (torch.acos(ct) - t0) ** 2).sum()
                fs = -torch.autograd.grad(ub + ua, y)[0]
            ub, ua = ub.detach(), ua.detach()
        usf = z
        if self.grid is not None and self.split:
            usf, fw = self.wall(x)
            fs = fs + fw
        return fs, torch.stack([ub, ua, z, z, ub + ua, vir, z])

    def mv2(self, v):
        return float((self.m * (v * v).sum(0)).sum())


def _exact_nve(E, x, v, fl, fs, dt, nin, K):
    lh, sh, kh = [], [], []
    for _ in range(K):
        v = v + dt / 2 * fl / E.m
        for _ in range(nin):
            v = v + dt / nin / 2 * fs / E.m
            x = x + dt / nin * v
            fs, ts = E.short(x)
            v = v + dt / nin / 2 * fs / E.m
        fl, tl = E.long(x)
        v = v + dt / 2 * fl / E.m
        lh.append(tl)
        sh.append(ts)
        kh.append(0.5 * E.mv2(v))
    return x, v, fl, fs, torch.stack(lh), torch.stack(sh), _t(kh)


def _implicit(E, v, f, p, q, dt, g, T):
    """v' = v + dt/2 (f/m - p' v'), p' = p + dt/2 (sum m v'^2 - g T) / q."""
    u = v + dt / 2 * f / E.m
    a = E.mv2(u)
    pn = p
    for _ in range(200):
        s = a / (1 + dt / 2 * pn) ** 2
        r = pn - p - dt / 2 * (s - g * T) / q
        step = r / (1 + dt / 2 * dt / q * s / (1 + dt / 2 * pn))
        pn -= step
        if abs(step) <= 1e-15 * abs(pn):
            break
    return u / (1 + dt / 2 * pn), pn, a / (1 + dt / 2 * pn) ** 2


def _exact_nvt(E, x, v, fl, fs, dt, nin, K, q, T, g):
    ps = pss = 0.0
    d = dt / nin
    for _ in range(K):
        v = v + dt / 2 * (fl / E.m - ps * v)
        for _ in range(nin):
            s2 = E.mv2(v)
            v = v + d / 2 * (fs / E.m - pss * v)
            x = x + d * v
            pss = pss + (s2 - g * T) * d / 2 / q
            fs, ts = E.short(x)
            v, pss, s2 = _implicit(E, v, fs, pss, q, d, g, T)
        ps = ps + (s2 - g * T) * dt / 2 / q
        fl, tl = E.long(x)
        v, ps, s2 = _implicit(E, v, fl, ps, q, dt, g, T)
    return x, v, fl, fs, tl, ts, s2 / 2


def _exact_npt(E, x, v, fl, fs, tl, ts, dt, nin, K, Qt, Qb, T, P, nf):
    vts = vbs = 0.0
    d, o = dt / nin, 1.0 + 3.0 / nf
    ukin = 0.0

    def op(v):
        nonlocal vts, vbs, ukin
        V = float(E.L.prod())
        m2 = E.mv2(v)
        pd = float(tl[11] + ts[5]) - 3.0 * P * V
        vts += dt / 4 * (m2 + Qb * vbs * vbs - (nf + 1) * T) / Qt
        B = math.exp(-vts * dt / 8)
        vbs = (vbs * B + dt / 4 * (o * m2 + pd) / Qb) * B
        A = math.exp(-dt / 2 * (vts + o * vbs))
        vbs *= B
        m2 *= A * A
        vbs = (vbs + dt / 4 * (o * m2 + pd) / Qb) * B
        vts += dt / 4 * (m2 + Qb * vbs * vbs - (nf + 1) * T) / Qt
        ukin = m2 / 2
        return v * A

    for _ in range(K):
        v = op(v) + dt / 2 * fl / E.m
        for _ in range(nin):
            A = math.exp(d / 2 * vbs)
            v = v + d / 2 * fs / E.m
            x = (x * A + d * v) * A
            E.L = E.L * math.exp(d * vbs)
            fs, ts = E.short(x)
            v = v + d / 2 * fs / E.m
        fl, tl = E.long(x)
        v = op(v + dt / 2 * fl / E.m)
    return x, v, fl, fs, tl, ts, ukin


def _exact_fit(case, systems):
    """Energies of the replicas and the loss's gradients, by autograd."""
    sets = _params(systems)
    eps, sig, q = (v.to(_t([0.0]).device).requires_grad_() for v in sets[0])
    pos, energy = [], []
    for s in systems:
        E = _Exact(s)
        x = _t(_xyz(s)).requires_grad_()
        pos.append(x)
        site = torch.arange(E.n, device=x.device) % 3
        with torch.no_grad():
            i, j = E.pairs(x)
        d = x[:, i] - x[:, j]
        d = d - E.L[:, None] * torch.round(d.detach() / E.L[:, None])
        r2 = (d * d).sum(0)
        qa = q[site]
        e = E._real(torch.sqrt(r2), E.C * qa[i] * qa[j])[0].sum()
        o = (site[i] == 0) & (site[j] == 0)
        s6 = (sig[0] ** 2 / r2[o]) ** 3
        e = e + (4 * eps[0] * (s6 * s6 - s6)).sum()
        for a, b in ((0, 1), (0, 2), (1, 2)):
            w = x[:, E.b2 + a] - x[:, E.b2 + b]
            r = torch.sqrt((w * w).sum(0))
            qq = E.C * q[a] * q[b]
            e = e + E._real(r, qq)[0].sum() - (qq / r).sum()
        self_c = E.kappa / math.sqrt(math.pi) + math.erfc(E.kappa * E.rc) / (2 * E.rc)
        energy.append(e - E.C * self_c * (qa * qa).sum())
    e = torch.stack(energy)
    loss = ((e + 20000.0 * case["mols"]) / 1e6).square().mean()
    g = torch.autograd.grad(loss, pos + [eps, sig, q])
    # positions: the engine gives minus the forces of the truncated sums
    return dict(energy=e.detach(), loss=loss.detach(), dpos=torch.cat(g[:-3], dim=1), deps=g[-3],
                dsig=g[-2], dq=g[-1])


def exact(case, seed):
    kind = case["kind"]
    if kind == "hmc":
        return None     # the chains follow the engine's own random streams
    systems = _systems(case, seed)
    if kind == "fit":
        return _exact_fit(case, systems)
    with torch.no_grad():
        if kind == "call":
            E = _Exact(systems[0])
            x = _t(_moved(systems[0], seed)[0])
            (fl, tl), (fs, ts) = E.long(x), E.short(x)
            return dict(fl=fl, fs=fs, long=tl, short=ts)
        vel, got, at = _t(_start_velocities(case, systems, seed)), [], 0
        for s in systems:
            E = _Exact(s)
            E.split = kind == "tube"
            x, v = _t(_xyz(s)), vel[:, at:at + s.natom]
            at += s.natom
            (fl, tl), (fs, ts) = E.long(x), E.short(x)
            dt, nin, K = s.delt, s.run.nstep_inner, case["steps"]
            nf = 3 * s.natom - s.run.nconstraint
            if kind in ("nve", "tube"):
                got.append(_exact_nve(E, x, v, fl, fs, dt, nin, K))
            elif kind in ("nvt", "nvt_argon"):
                q = 4.0 * nf if kind == "nvt" else 100.0 * s.natom / 864.0
                got.append(_exact_nvt(E, x, v, fl, fs, dt, nin, K, q, s.treq, nf))
            else:
                got.append(_exact_npt(E, x, v, fl, fs, tl, ts, dt, nin, K, 4.0 * nf, 400.0 * nf,
                                      s.treq, s.preq, nf))
        out = {k: torch.cat([g[i] for g in got], dim=1)
               for i, k in enumerate(("pos", "vel", "fl", "fs"))}
        if kind in ("nve", "tube"):
            lh, sh, kh = (torch.stack([g[i] for g in got], dim=1) for i in (4, 5, 6))
            out.update(lhist=lh, shist=sh, khist=kh.reshape(-1), long=lh[-1], short=sh[-1],
                       ukin=kh[-1])
        else:
            out.update(long=got[0][4][None], short=got[0][5][None], ukin=_t([got[0][6]]))
        return out
