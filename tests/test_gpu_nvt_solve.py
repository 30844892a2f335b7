"""The NVT step's substep kernels (k_nvt.hip) on every path that their
dispatch takes and at the edges of their workgroups, against the CPU
restatement of vver_nh_3 (tests/md_cpu.py): single sites (256 per
workgroup), molecules of up to three and four sites and terms (64 per
workgroup), and larger ones, which go by atoms (256 per workgroup).

Two steps of two or more substeps in FP64.  Bounds as in test_gpu_md.py:
positions and velocities within 1e-9 relative (a Newton pass more or less
moves the thermostat momentum by up to 1e-10 of itself), the momenta within
1e-8 of their scale."""
import numpy as np
import pytest

from mspms2_amd import configs
from mspms2_amd.engine import LONG_TERMS_BYTES, SHORT_TERMS_BYTES, Engine
from tests.md_cpu import NvtCpu
from tests.util import system_of

pytestmark = pytest.mark.gpu


def _water(nmol):
    return configs.water_box(n_side=5, L=5 * 3.104, rc=7.0, kappa=0.35, kmax=5, ksqmax=25,
                             nmol=nmol, seed=40 + nmol)


def _chain(nmol):
    """Four sites and four terms: butane with one angle and no dihedral."""
    rd = configs.butane_box(nmol=nmol)
    rd.species[0].angles = rd.species[0].angles[:1]
    rd.species[0].dihedrals = []
    return rd


CASES = {
    "argon-256": lambda: [configs.lj_fcc(ncell=4, jitter=0.04, seed=5)],        # one full block
    "argon-500": lambda: [configs.lj_fcc(ncell=5, jitter=0.04, seed=6)],
    "water-63": lambda: [_water(63)],
    "water-64": lambda: [_water(64)],
    "water-65": lambda: [_water(65)],
    "water-batch": lambda: [_water(1), _water(65), _water(125)],
    "mixture": lambda: [configs.mixture_box(n_water=70, n_co=30, L=20.0)],      # a Morse bond
    "chain-65": lambda: [_chain(65)],
    "butane-64": lambda: [configs.butane_box(nmol=64)],                         # 6 terms: by atoms
    "zoo-43": lambda: [configs.bonded_zoo(nmole=43)],                           # 258 atoms
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("inner", [1, 3])
def test_nvt_substeps_match_restatement(name, inner):
    import torch
    rds = CASES[name]()
    print(f"case {name} inner={inner}", flush=True)
    for rd in rds:
        rd.run.nstep_inner = inner
        rd.run.delt *= 0.25
    systems = [system_of(rd) for rd in rds]
    rng = np.random.default_rng(9)
    v0s = [rng.standard_normal((3, s.natom)) * np.sqrt(s.treq / s.masses()) for s in systems]
    qs = [4.0 * s.natom for s in systems]
    refs = []
    for s, v0, q in zip(systems, v0s, qs):
        c = NvtCpu(s, v0, q, 0.5 * q)
        c.step()
        c.step()
        refs.append(c)
    eng = Engine.replicas(systems, precision="fp64")
    eng.nvt_set(qs, [0.5 * q for q in qs], [s.treq for s in systems],
                [3 * s.natom - 3 for s in systems])
    dev = torch.device("cuda:0")
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=dev).contiguous()  # noqa: E731
    x0 = eng.packed_positions()
    pos, vel, fl, fs = t(x0), t(eng.pack(v0s)), t(eng.frclong()[0]), t(eng.frcshort()[0])
    lt = torch.zeros(eng.nrep * LONG_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    st = torch.zeros(eng.nrep * SHORT_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    uk = torch.zeros(eng.nrep, dtype=torch.float64, device=dev)
    torch.cuda.synchronize()
    eng.nvt_run_device(pos, vel, fl, fs, systems[0].delt, inner, 2, lt, st, uk, graph=False)
    torch.cuda.synchronize()
    eng.sync()
    states = eng.nvt_get()
    terms = st.cpu().numpy().reshape(eng.nrep, -1)
    x, v = eng.unpack(pos.cpu().numpy()), eng.unpack(vel.cpu().numpy())
    eng.close()
    for r, c in enumerate(refs):
        for got, ref in ((x[r], c.x), (v[r], c.v)):
            assert np.linalg.norm(got - ref) <= 1e-9 * np.linalg.norm(ref)
        for k in ("ps", "pss", "ss", "sss"):
            ref = getattr(c, k)
            assert abs(states[r][k] - ref) <= 1e-8 * max(abs(ref), 1e-3), (r, k)
        assert abs(states[r]["ukin"] - c.ukin) <= 1e-9 * c.ukin
        # uintra of the last substep
        ref = c.o.frcshort(*c.x)[1]["uintra"]
        assert abs(terms[r][4] - ref) <= 1e-8 * max(abs(ref), 1.0)
