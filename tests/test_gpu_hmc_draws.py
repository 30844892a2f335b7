"""The velocity draws of a whole workgroup (k_hmc.hip draw_velocities) against
the one-by-one draws of the CPU restatement: odd and even component counts
(the second Gaussian of the last pair is kept for the next velinit), one
block of draws and several, a single molecule; streams left bit for bit where
the restatement leaves them.  Velocities within 1e-13 as in test_gpu_hmc.py
(log and sqrt are the only operations that are not exact)."""
import numpy as np
import pytest

from mspms2_amd import configs
from mspms2_amd.engine import LONG_TERMS_BYTES, SHORT_TERMS_BYTES, Engine
from tests.hmc_cpu import HmcChain
from tests.util import system_of

pytestmark = pytest.mark.gpu


def test_draws_match_restatement_over_moves():
    import torch
    dev = torch.device("cuda:0")
    sizes = [1, 2, 27, 64, 125]          # 9 to 1125 components, odd and even
    systems = [system_of(configs.water_box(n_side=5, L=5 * 3.104, rc=6.0, kappa=0.35, kmax=3,
                                           ksqmax=9, nmol=n, seed=60 + n)) for n in sizes]
    nr = len(systems)
    ij, kl = [31 + 7 * r for r in range(nr)], [17 + 5 * r for r in range(nr)]
    eng = Engine.replicas(systems, precision="fp64")
    pos = torch.tensor(eng.packed_positions(), device=dev)
    vel, fl, fs = (torch.zeros_like(pos) for _ in range(3))
    new = lambda n: torch.zeros(n, dtype=torch.float64, device=dev)  # noqa: E731
    lt, st, uk = new(nr * LONG_TERMS_BYTES // 8), new(nr * SHORT_TERMS_BYTES // 8), new(nr)
    print(f"case draws {sizes}", flush=True)
    eng.hmc_init(ij, kl, [s.treq for s in systems], 0, vel)
    chains = [HmcChain(s, a, b) for s, a, b in zip(systems, ij, kl)]
    delt = 0.1 * systems[0].delt
    for move in range(4):
        torch.cuda.synchronize()
        for r, (c, v) in enumerate(zip(chains, eng.unpack(vel.cpu().numpy()))):
            if move == 0:
                assert np.abs(v - c.v).max() <= 1e-13 * np.abs(c.v).max()
        eng.hmc_run_device(pos, vel, fl, fs, delt, 2, 1, 1, lt, st, uk, graph=False)
        torch.cuda.synchronize()
        _, _, dh = eng.hmc_stats()
        for r, c in enumerate(chains):
            _, ref = c.move(delt, 2, 1)
            assert abs(dh[r] - ref) <= 1e-7 * max(abs(ref), 1e-3), (move, r, dh[r], ref)
    eng.sync()
    for r, c in enumerate(chains):
        assert np.abs(eng.unpack(pos.cpu().numpy())[r] - c.x).max() <= 1e-8
        assert np.array_equal(eng.hmc_draw(r, 101), c.g.rng.next(101))
    eng.close()


def test_long_draw_matches_restatement():
    """2048 atoms: 6144 components, about eight blocks of draws."""
    import torch
    s = system_of(configs.lj_fcc(ncell=8, jitter=0.02, seed=3))
    eng = Engine.replicas([s], precision="mixed")
    vel = torch.zeros((3, s.natom), dtype=torch.float64, device="cuda:0")
    print(f"case draws {s.natom} atoms", flush=True)
    eng.hmc_init([5], [9], [s.treq], 0, vel)
    torch.cuda.synchronize()
    c = HmcChain(s, 5, 9)
    assert np.abs(vel.cpu().numpy() - c.v).max() <= 1e-13 * np.abs(c.v).max()
    assert np.array_equal(eng.hmc_draw(0, 500), c.g.rng.next(500))
    eng.close()
