"""The harmonic bond and angle of the device integrators' inner loops
(inner_terms.h), which all of NVE, NVT and NPT take: no further from the exact
forces (80-bit arithmetic, at the positions that the step reached) than the
reference's own expressions in 64 bits are, and finite on straight molecules,
whose cosine may round beyond 1."""
import numpy as np
import pytest

from mspms2_amd import abi, configs
from mspms2_amd.engine import LONG_TERMS_BYTES, SHORT_TERMS_BYTES, Engine
from mspms2_amd.runio import RunDir, RunInput, Site, SpeciesSpec
from mspms2_amd.system import System
from oracle.oracle import Oracle
from tests.util import system_of

pytestmark = pytest.mark.gpu


def _step(s, kind, v0, inner, delt):
    """One outer step: positions and short forces, (3, N)."""
    import torch
    dev = torch.device("cuda:0")
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=dev).contiguous()  # noqa: E731
    x0 = np.stack([s.xx, s.yy, s.zz])
    pos, vel, fl, fs = t(x0), t(v0), t(np.zeros_like(x0)), t(np.zeros_like(x0))
    lt = torch.zeros(LONG_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    st = torch.zeros(SHORT_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    uk = torch.zeros(1, dtype=torch.float64, device=dev)
    eng = Engine(s, precision="fp64")
    call = eng.vver_run_device
    if kind == "nvt":
        eng.nvt_set(400.0 * s.natom, 400.0 * s.natom, s.treq, 3 * s.natom)
        call = eng.nvt_run_device
    elif kind == "npt":
        eng.npt_set(300.0 * s.natom, 30000.0 * s.natom, s.treq, 0.0, 3 * s.natom, vts=0.0, vbs=0.0)
        call = eng.npt_run_device
    torch.cuda.synchronize()
    call(pos, vel, fl, fs, delt, inner, 1, lt, st, uk, graph=False)
    eng.sync()
    eng.close()
    return pos.cpu().numpy(), fs.cpu().numpy(), st.cpu().numpy()


def _exact(s, x):
    """Bond and angle forces of three-site water in 80 bits."""
    q, sp = np.longdouble, s.species[0]
    X = x.astype(q).reshape(3, -1, 3)            # axis, molecule, site
    f = np.zeros_like(X)
    for (i, j), para in zip(sp.bnd_idx, sp.bnd_para):
        d = X[:, :, i] - X[:, :, j]
        r = np.sqrt((d * d).sum(0))
        g = -q(para[0]) * (r - q(para[1])) / r * d
        f[:, :, i] += g
        f[:, :, j] -= g
    (a, b, c), para = sp.agl_idx[0], sp.agl_para[0]
    u, v = X[:, :, a] - X[:, :, b], X[:, :, c] - X[:, :, b]
    ru, rv = np.sqrt((u * u).sum(0)), np.sqrt((v * v).sum(0))
    u, v = u / ru, v / rv
    cost = (u * v).sum(0)
    gam = q(para[0]) * (np.arccos(cost) - q(para[1])) / np.sqrt(1 - cost * cost)
    fa, fc = gam * (v - u * cost) / ru, gam * (u - v * cost) / rv
    f[:, :, a] += fa
    f[:, :, c] += fc
    f[:, :, b] -= fa + fc
    return f.reshape(3, -1)


@pytest.mark.parametrize("kind", ["nve", "nvt", "npt"])
def test_no_further_from_exact_than_the_reference(kind):
    s = system_of(configs.water_box(n_side=10, L=31.04, rc=9.0, kappa=0.3, kmax=3, ksqmax=9,
                                    seed=4))
    d = 0.04 / s.params["sigma_base"]
    rng = np.random.default_rng(6)
    for v in (s.xx, s.yy, s.zz):
        v += rng.uniform(-d, d, v.shape)
    print(f"case {kind} natom={s.natom}", flush=True)
    x, g, _ = _step(s, kind, np.zeros((3, s.natom)), 1, 1e-9)
    want = _exact(s, x)
    ref, _ = Oracle(s).frcshort(*x)
    err = [float(np.linalg.norm((np.asarray(f, dtype=np.longdouble) - want).astype(np.float64)))
           for f in (g, ref)]
    scale = float(np.linalg.norm(want.astype(np.float64)))
    print(f"{kind}: RMS error of the norm, engine {err[0] / scale:.2e}, reference's "
          f"expressions {err[1] / scale:.2e}", flush=True)
    assert err[1] <= 1e-14 * scale        # the two agree on what is computed
    assert err[0] <= err[1]


@pytest.mark.parametrize("kind", ["nve", "nvt", "npt"])
def test_straight_molecules(kind):
    """2,000 straight three-site molecules along the z axis, of bond lengths
    drawn around the force field's, moving along it."""
    n, rng = 2000, np.random.default_rng(8)
    site = lambda name, z: Site(type=0, name=name, xx=0.0, yy=0.0, zz=z, aw=0.014,  # noqa: E731
                                epsilon=0.0, sigma=3.0, charge=0.0, ghost_type=1)
    sp = SpeciesSpec(name="rod", nmole=n, sites=[site("A", -1.16), site("B", 0.0), site("A", 1.16)],
                     bonds=[(i, i + 1, abi.BOND_HARMONIC, 2.0e5, 1.16, 0.0) for i in (0, 1)],
                     angles=[(0, 1, 2, abi.ANGLE_HARMONIC, 4.0e4, np.pi, 0.0, 0.0, 0.0)])
    L = 200.0
    o = rng.uniform(0.0, L, (n, 1, 3))
    z = np.zeros((n, 3, 3))
    z[:, 0, 2], z[:, 2, 2] = -1.16 * rng.uniform(0.93, 1.07, n), 1.16 * rng.uniform(0.93, 1.07, n)
    run = RunInput(boxlx=L, boxly=L, boxlz=L, rcuton=9.0, rcutoff=9.0, rcutoffelec=9.0,
                   treq=300.0, iChargeType=abi.ELEC_NONE, delt=1.0)
    s = System.from_rundir(RunDir(run=run, sysname="rods", species=[sp],
                                  xyz=(o + z).reshape(-1, 3)))
    v0 = np.zeros((3, s.natom))
    v0[2] = rng.standard_normal(s.natom) * np.sqrt(s.treq / s.masses())
    print(f"case straight {kind}", flush=True)
    x, g, st = _step(s, kind, v0, 2, s.delt)
    assert np.isfinite(x).all() and np.isfinite(g).all() and np.isfinite(st).all()
    ref, _ = Oracle(s).frcshort(*x)
    assert np.isfinite(ref).all()
    # the angle adds forces of K 1e-16 / 1e-8 1e-8 along the axis
    assert np.linalg.norm(g - ref) <= 1e-11 * np.linalg.norm(ref)
