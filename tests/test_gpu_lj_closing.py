"""The closing pass of an NVE step of an LJ fluid (no charges, no molecules),
whose slot forces and half kick the finalize kernel adds while replicas are
small (one sweep of its 16,384 threads, two, four) and launches of their own
for larger ones, one large replica among small ones being enough: velocities
and kinetic energy from the step's own forces, forces and energies against a
force call at the positions reached.

The kicks are three roundings of numbers of the velocities' size (1e-14 of the
norm); the sums of the two force evaluations may differ in order (1e-12)."""
import numpy as np
import pytest

from mspms2_amd import configs
from mspms2_amd.engine import LONG_TERMS_BYTES, SHORT_TERMS_BYTES, Engine
from tests.util import system_of

pytestmark = pytest.mark.gpu

# cells per edge of the replicas: 4 n^3 sites each
CASES = {"256": [4], "batch": [4, 7, 5], "16384": [16], "19652": [17], "62500": [25],
         "70304": [26], "batch-70304": [4, 26]}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_step_closes_with_its_own_forces(name, precision):
    import torch
    systems = [system_of(configs.lj_fcc(ncell=k, jitter=0.05, seed=k)) for k in CASES[name]]
    rng, dev = np.random.default_rng(3), torch.device("cuda:0")
    print(f"case {name} {precision} natom={sum(s.natom for s in systems)}", flush=True)
    eng = Engine.replicas(systems, precision=precision)
    eng.set_list_skin(0.3)
    m = np.concatenate([s.masses() for s in systems])
    x0 = eng.packed_positions()
    v0 = rng.standard_normal(x0.shape) * np.sqrt(systems[0].treq / m)
    f0, _ = eng.frclong(*x0)
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=dev).contiguous()  # noqa: E731
    pos, vel, fl, fs = t(x0), t(v0), t(f0), t(np.zeros_like(x0))
    nr = len(systems)
    lt = torch.zeros((nr, LONG_TERMS_BYTES // 8), dtype=torch.float64, device=dev)
    st = torch.zeros((nr, SHORT_TERMS_BYTES // 8), dtype=torch.float64, device=dev)
    uk = torch.zeros(nr, dtype=torch.float64, device=dev)
    dt = systems[0].delt
    torch.cuda.synchronize()
    eng.vver_run_device(pos, vel, fl, fs, dt, 1, 1, lt, st, uk, graph=False)
    eng.sync()
    x, v, f = (b.cpu().numpy() for b in (pos, vel, fl))
    half = v0 + 0.5 * dt * f0 / m
    assert np.linalg.norm(x - (x0 + dt * half)) <= 1e-14 * np.linalg.norm(x)
    want = half + 0.5 * dt * f / m
    assert np.linalg.norm(v - want) <= 1e-14 * np.linalg.norm(v)
    g, terms = eng.frclong(*x)
    terms = [terms] if nr == 1 else terms
    assert np.linalg.norm(f - g) <= 1e-12 * np.linalg.norm(g)
    for r, (w, mm) in enumerate(zip(eng.unpack(v), eng.unpack(m[None]))):
        ke = 0.5 * (mm * w * w).sum()
        assert abs(float(uk[r]) - ke) <= 1e-12 * ke
        assert abs(float(lt[r, 0]) - terms[r]["uvdw"]) <= 1e-12 * abs(terms[r]["uvdw"])
    eng.close()
