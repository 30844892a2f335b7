"""The Ewald reciprocal kernels (k_recip.hip) on every tile count their
dispatch takes: kz tiles of 8 (kmaxz 8, 9 and 16), row tiles of 8 shared by
up to 8 waves (1, 2, 4, 7 and 9 tiles a wave), 32- and 64-atom force groups,
one and several 64-atom tables per chunk, axes without k, replicas of
different KMAX; against a direct sum in numpy.

The systems are three-site ions with a 0.2 A cutoff, shorter than any
distance in them, so that forces and energy are the reciprocal part alone.
Bound 1e-11 of the norm: the powers exp(i n t) by repeated products are off
by up to 16 ulp (4e-15), and random charges leave S(k) about sqrt(N) of its
N terms, a factor of up to 260 here."""
import numpy as np
import pytest

from mspms2_amd import abi, configs
from mspms2_amd.engine import Engine
from mspms2_amd.runio import RunDir, RunInput
from mspms2_amd.system import System

pytestmark = pytest.mark.gpu


def _system(nmol, kmax, ksq, seed=1, q=(-0.8, 0.5, 0.3)):
    rng = np.random.default_rng(seed)
    L = np.array([1.0, 1.1, 0.97]) * 3.2 * np.ceil(max(nmol, 27) ** (1.0 / 3.0) - 1e-9)
    sp = configs.water_species(nmol)
    for s, v in zip(sp.sites, q):
        s.charge, s.epsilon, s.ghost_type = v, 0.0, 1
    t = np.array([[s.xx, s.yy, s.zz] for s in sp.sites])
    # a lattice of 3 A or more, moved by up to 0.3 A, sites in and out of the box
    # (the engine takes unwrapped positions)
    n = int(np.ceil(max(nmol, 27) ** (1.0 / 3.0) - 1e-9))
    g = np.stack(np.meshgrid(*(np.arange(n),) * 3, indexing="ij"), -1).reshape(-1, 3)
    g = g[rng.permutation(len(g))[:nmol]] / n + rng.integers(-1, 2, (nmol, 3))
    xyz = (g[:, None] * L + t + rng.uniform(-0.3, 0.3, (nmol, 1, 3))).reshape(-1, 3)
    run = RunInput(boxlx=L[0], boxly=L[1], boxlz=L[2], rcuton=0.2, rcutoff=0.2, rcutoffelec=0.2,
                   iChargeType=abi.ELEC_EWALD, kappa=0.35, kmaxx=kmax[0], kmaxy=kmax[1],
                   kmaxz=kmax[2], ksqmax=ksq, fEwald_BC=abi.EWALD_BC_TINFOIL, treq=300.0)
    return System.from_rundir(RunDir(run=run, sysname="ions", species=[sp], xyz=xyz))


def _direct(s):
    """ufourier, forces and dU/dq per atom: the sum over all k, one by one
    (src/frclong.c:988-1048)."""
    p = s.params
    L = np.array([p["boxlx"], p["boxly"], p["boxlz"]])
    x, q = np.stack([s.xx, s.yy, s.zz]), s.charges()
    C = 167100.80840 / p["epsilon_base"] / p["sigma_base"]
    vf = 2.0 * np.pi / L.prod()
    u, f, dq = 0.0, np.zeros_like(x), np.zeros(s.natom)
    for kx in range(0, p["kmaxx"] + 1):
        for ky in range(-p["kmaxy"], p["kmaxy"] + 1):
            for kz in range(-p["kmaxz"], p["kmaxz"] + 1):
                n2 = kx * kx + ky * ky + kz * kz
                if not 0 < n2 <= p["ksqmax"] or (kx, ky, kz) < (0, 0, 0):
                    continue
                k = 2.0 * np.pi * np.array([kx, ky, kz]) / L
                w = 2.0 * np.exp(-(k @ k) / (4.0 * p["kappa"] ** 2)) / (k @ k)
                e = np.exp(1j * (k @ x))
                S = (q * e).sum()
                u += w * abs(S) ** 2
                g = 2.0 * vf * C * w * np.conj(S) * e
                dq += g.real
                f += q * g.imag * k[:, None]
    return u * vf * C, f, dq, C


CASES = [(11, (3, 3, 3), 9), (21, (8, 8, 8), 64), (22, (5, 2, 8), 64), (64, (2, 7, 9), 81),
         (43, (16, 16, 16), 256), (10, (16, 16, 16), 768), (20, (0, 4, 3), 16),
         (20, (4, 0, 5), 25), (20, (3, 3, 0), 9), (20, (0, 0, 1), 1), (1, (6, 6, 16), 256),
         (11200, (3, 3, 3), 9), (22000, (2, 2, 2), 4), (22000, (1, 1, 9), 81)]


def _check(s, fl, t):
    u, f, _, _ = _direct(s)
    assert abs(t["ufourier"] - u) <= 1e-11 * abs(u), (t["ufourier"], u)
    assert np.linalg.norm(fl - f) <= 1e-11 * np.linalg.norm(f)


@pytest.mark.parametrize("nmol,kmax,ksq", CASES)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_reciprocal_matches_direct_sum(nmol, kmax, ksq, precision):
    s = _system(nmol, kmax, ksq)
    print(f"case nmol={nmol} kmax={kmax} ksqmax={ksq} {precision}", flush=True)
    eng = Engine(s, precision=precision)
    fl, t = eng.frclong()
    eng.close()
    _check(s, fl, t)


def test_reciprocal_of_replicas_with_different_kmax():
    shapes = [(30, (3, 4, 5), 25), (1, (2, 2, 2), 12), (70, (8, 3, 12), 144), (5, (9, 16, 1), 200)]
    systems = [_system(n, k, q, seed=3 + i) for i, (n, k, q) in enumerate(shapes)]
    print("case replicas", flush=True)
    eng = Engine.replicas(systems, precision="fp64")
    f, terms = eng.frclong()
    parts = eng.unpack(f)
    eng.close()
    for s, fl, t in zip(systems, parts, terms):
        _check(s, fl, t)


def test_reciprocal_of_many_small_replicas():
    """180 replicas of up to five 64-atom tables, more than 512 tables in all:
    chunks of several tables, most of them a whole replica."""
    systems = [_system(20 + 7 * (r % 12), (3, 2, 3), 9, seed=r) for r in range(180)]
    assert sum((s.natom + 63) // 64 for s in systems) > 512
    print("case many replicas", flush=True)
    eng = Engine.replicas(systems, precision="fp64")
    f, terms = eng.frclong()
    parts = eng.unpack(f)
    eng.close()
    for s, fl, t in zip(systems, parts, terms):
        _check(s, fl, t)


@pytest.mark.parametrize("nmol,kmax,ksq", [(40, (5, 6, 7), 49), (33, (6, 5, 11), 150),
                                           (22000, (1, 1, 9), 81)])
def test_charge_derivative_matches_direct_sum(nmol, kmax, ksq):
    s = _system(nmol, kmax, ksq)
    print(f"case adjoint nmol={nmol} kmax={kmax}", flush=True)
    eng = Engine(s, precision="fp64")
    fl, t, g = eng.param_grad()
    eng.close()
    _check(s, fl, t)
    _, _, dq, C = _direct(s)
    q = s.charges()
    dq = dq - 2.0 * C * s.params["kappa"] / np.sqrt(np.pi) * q  # the self energy
    ref = dq.reshape(-1, 3).sum(0)
    assert np.abs(g["charge"][0] - ref).max() <= 1e-11 * np.abs(dq).sum()
