"""Rounding error of the exact mode's electrostatic pair terms: boxes of two
ions each, whose energies and forces are one pair's, against 40-digit
arithmetic.  A term is a product of about ten factors that are each within an
ulp (2^-53 / sqrt(3) RMS per rounding): an RMS of about 2.5e-16.  erfc and
exp(-x^2) amplify an error of their argument by 2 x^2, 16 at the largest x
here: an argument that is a square root and a product, each rounded once,
would give 7e-16.  Bound 4e-16."""
from decimal import Decimal, getcontext

import numpy as np
import pytest

from mspms2_amd import abi
from mspms2_amd.engine import Engine
from mspms2_amd.runio import RunDir, RunInput, Site, SpeciesSpec
from mspms2_amd.system import System
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

KAPPA, L, RC = 0.28, 24.0, 10.0
NPAIR = 400


def ions(xyz, elec="ewald", q=(1.0, -1.0)):
    """Single-site ions without LJ terms (GHOST_LJ) at xyz (Angstrom)."""
    sp = [SpeciesSpec(name=f"ion{k}", nmole=1, sites=[
        Site(type=k, name="I", xx=0.0, yy=0.0, zz=0.0, aw=0.02, epsilon=0.0, sigma=3.0, charge=v,
             ghost_type=1, interp_type=0)]) for k, v in enumerate(q)]
    run = RunInput(boxlx=L, boxly=L, boxlz=L, rcuton=RC, rcutoff=RC, rcutoffelec=RC, treq=300.0,
                   iChargeType=abi.ELEC_EWALD if elec == "ewald" else abi.ELEC_WOLF, kappa=KAPPA,
                   kmaxx=0, kmaxy=0, kmaxz=1, ksqmax=1, fEwald_BC=abi.EWALD_BC_TINFOIL)
    return System.from_rundir(RunDir(run=run, sysname="ions", species=sp,
                                     xyz=np.asarray(xyz, dtype=np.float64)))


def _pi():
    # Machin's formula
    def atan_inv(n):
        t, s, k, sign = Decimal(1) / n, Decimal(0), 1, 1
        while t > Decimal(10) ** -48:
            s += sign * t / k
            t /= n * n
            k += 2
            sign = -sign
        return s
    return 4 * (4 * atan_inv(5) - atan_inv(239))


def _erfc(x, pi):
    """1 - 2 x / sqrt(pi) exp(-x^2) sum (2 x^2)^k / (2 k + 1)!!: positive
    terms only, and 1 - erf loses 4 of 50 digits at x = 3."""
    s = t = Decimal(1)
    k = 0
    while t > s * Decimal(10) ** -48:
        k += 1
        t *= 2 * x * x / (2 * k + 1)
        s += t
    return 1 - 2 * x / pi.sqrt() * (-x * x).exp() * s


def _pairs():
    rng = np.random.default_rng(12)
    out = []
    while len(out) < NPAIR:
        d = rng.uniform(-RC, RC, 3)
        if 2.0 < np.linalg.norm(d) < RC - 0.01:
            out.append(np.stack([np.full(3, 12.0), 12.0 + d]))
    return out


@pytest.mark.parametrize("elec", ["ewald", "wolf"])
def test_pair_terms_against_40_digits(elec):
    getcontext().prec = 50
    pi = _pi()
    systems = [ions(x, elec) for x in _pairs()]
    print(f"case {elec}, {NPAIR} boxes of two ions", flush=True)
    eng = Engine.replicas(systems, precision="fp64")
    f, terms = eng.frclong()
    parts, P = eng.unpack(f), eng.params
    eng.close()
    eu, ef = [], []
    for s, g, t in zip(systems, parts, terms):
        d = [np.float64(v[0]) - np.float64(v[1]) for v in (s.xx, s.yy, s.zz)]
        rsq = Decimal(float(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]))  # as the engine rounds it
        q = [Decimal(float(v)) for v in s.charges()]
        kap, cq = Decimal(P.kappa), Decimal(P.coulomb_prefactor) * q[0] * q[1]
        r = rsq.sqrt()
        ec, ex = _erfc(kap * r, pi), (-kap * kap * rsq).exp()
        if elec == "ewald":
            # (the force of these boxes has a reciprocal part; it is looked at
            # under Wolf)
            u = cq * ec / r
            eu.append(float((Decimal(t["ureal"]) - u) / u))
            continue
        # relative to the terms that cancel near the cutoff
        v1, v2, f1, f2 = (Decimal(v) for v in (P.wolfvcon1, P.wolfvcon2, P.wolffcon1, P.wolffcon2))
        u = cq * (ec / r + v1 + v2 * (r - Decimal(P.rcutoffelec)))
        eu.append(float((Decimal(t["ureal"]) - u) / (cq * ec / r)))
        k = int(np.argmax(np.abs(d)))
        x, near = Decimal(float(d[k])), ec / rsq + f1 * ex / r
        ef.append(float((Decimal(float(g[k][0])) - cq / r * (near + f2) * x) / (cq / r * near * x)))
    rms = [float(np.sqrt(np.mean(np.square(e)))) for e in (eu, ef) if e]
    print(f"RMS relative error {elec}: " + ", ".join(f"{v:.2e}" for v in rms), flush=True)
    assert max(rms) <= 4e-16, rms


@pytest.mark.parametrize("elec", ["ewald", "wolf"])
def test_sites_on_one_point(elec):
    """Two charged sites on one point: the energy is infinite, with the sign of
    the charges' product, as the reference's C q q / r gives it (a sampling
    program rejects on it); the force has no value."""
    for q in ((1.0, -1.0), (1.0, 0.5)):
        s = ions([[3.0, 4.0, 5.0], [3.0, 4.0, 5.0]], elec, q)
        _, want = Oracle(s).frclong()
        print(f"case coincident {elec} {q}", flush=True)
        eng = Engine(s, precision="fp64")
        _, t = eng.frclong()
        eng.close()
        assert want["ureal"] == np.copysign(np.inf, q[0] * q[1])
        assert t["n_elec_pairs"] == want["n_elec_pairs"] == 1
        for k in ("ureal", "uelec", "uinter", "virial_inter"):
            assert np.array_equal(t[k], want[k], equal_nan=True), (k, t[k], want[k])
