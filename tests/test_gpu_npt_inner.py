"""The NPT step (k_npt.hip, and the inner loop in one launch of
k_integrate.hip) on every path that its dispatch takes -- single sites,
molecules of up to three and four sites and terms, four sites and
six terms, larger ones -- at the edges
of their workgroups and where a replica has more atoms than its workgroup
keeps in registers (4,096), against the CPU restatement of npt_respa
(tests/md_cpu.py).  Two steps in FP64 with the bounds of test_gpu_md.py."""
import numpy as np
import pytest

from mspms2_amd import configs
from mspms2_amd.engine import LONG_TERMS_BYTES, SHORT_TERMS_BYTES, Engine
from tests.md_cpu import NptCpu
from tests.test_gpu_md import rel
from tests.test_gpu_nvt_solve import _chain, _water
from tests.util import system_of

pytestmark = pytest.mark.gpu

CASES = {
    "argon-500": lambda: [configs.lj_fcc(ncell=5, jitter=0.04, seed=6)],
    "argon-5324": lambda: [configs.lj_fcc(ncell=11, jitter=0.04, seed=6)],
    "water-64": lambda: [_water(64)],
    "water-batch": lambda: [_water(1), _water(65), _water(125)],
    "chain-65": lambda: [_chain(65)],
    "butane-64": lambda: [configs.butane_box(nmol=64)],
    "butane-65": lambda: [configs.butane_box(nmol=65)],
    "zoo-43": lambda: [configs.bonded_zoo(nmole=43)],       # a launch per inner step
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("inner", [1, 3])
def test_npt_steps_match_restatement(name, inner):
    import torch
    rds = CASES[name]()
    print(f"case {name} inner={inner}", flush=True)
    for rd in rds:
        rd.run.nstep_inner = inner
        rd.run.delt *= 0.25
        rd.run.isLJlrcOn = 0
    systems = [system_of(rd) for rd in rds]
    rng = np.random.default_rng(9)
    v0s = [rng.standard_normal((3, s.natom)) * np.sqrt(s.treq / s.masses()) for s in systems]
    qt = [300.0 * 3 * s.natom for s in systems]
    qb = [3000.0 * 3 * s.natom for s in systems]
    refs = []
    for s, v0, a, b in zip(systems, v0s, qt, qb):
        c = NptCpu(s, v0, a, b, 0)
        c.step()
        c.step()
        refs.append(c)
    eng = Engine.replicas(systems, precision="fp64")
    eng.npt_set(qt, qb, [s.treq for s in systems], [s.preq for s in systems],
                [3 * s.natom for s in systems])
    dev = torch.device("cuda:0")
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=dev).contiguous()  # noqa: E731
    pos, vel = t(eng.packed_positions()), t(eng.pack(v0s))
    fl, fs = torch.zeros_like(pos), torch.zeros_like(pos)
    lt = torch.zeros(eng.nrep * LONG_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    st = torch.zeros(eng.nrep * SHORT_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    uk = torch.zeros(eng.nrep, dtype=torch.float64, device=dev)
    torch.cuda.synchronize()
    eng.frclong_device(pos, fl, lt)
    eng.frcshort_device(pos, fs, st)
    eng.sync()
    eng.npt_run_device(pos, vel, fl, fs, systems[0].delt, inner, 2, lt, st, uk, graph=False)
    torch.cuda.synchronize()
    eng.sync()
    xs, vs, states = eng.unpack(pos.cpu().numpy()), eng.unpack(vel.cpu().numpy()), eng.npt_get()
    eng.close()
    for c, x, v, state in zip(refs, xs, vs, states):
        assert rel(x, c.x) <= 1e-9 and rel(v, c.v) <= 1e-9
        assert np.allclose(state["boxl"], c.box, rtol=1e-12, atol=0)
        for k in ("vts", "vbs", "rts", "utsbs", "pinst", "ukin"):
            ref = getattr(c, k)
            assert abs(state[k] - ref) <= 1e-8 * max(abs(ref), 1e-3), (k, state[k], ref)
