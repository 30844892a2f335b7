"""The FP64 pair kernel (k_pair) where its queues and its erfc can go wrong:
cutoffs of half the box (nearly every lane of an entry in range, ambiguous
images), different LJ and electrostatic cutoffs, arguments of erfc from
nearly 0 to 18, LJ alone, Wolf, ghosts, and every number of waves per
i-cluster; pair counts and hashes equal to the oracle's, forces within 1e-12
of the norm and energies within 1e-12 of the pair energies' scale (the
oracle's own terms are good to a few 1e-16 each, sums of 1e4 to 1e5 of them
to about 1e-14)."""
import numpy as np
import pytest

from mspms2_amd import configs
from mspms2_amd.engine import Engine
from oracle.oracle import Oracle
from tests.util import system_of

pytestmark = pytest.mark.gpu


def _water(n, rc, rce, kappa, elec="ewald", seed=3):
    L = n * 3.104
    rd = configs.water_box(n_side=n, L=L, rc=min(rc, 0.5 * L), kappa=kappa, kmax=2, ksqmax=4,
                           elec=elec, seed=seed)
    rd.run.rcutoffelec = min(rce, 0.5 * L)
    return rd


CASES = {
    "half-box": lambda: _water(4, 99.0, 99.0, 0.3),
    "half-box-small": lambda: _water(3, 99.0, 99.0, 0.3),
    "lj-shorter": lambda: _water(5, 3.5, 7.5, 0.3),
    "lj-longer": lambda: _water(5, 7.5, 4.0, 0.3),
    "kappa-small": lambda: _water(4, 6.0, 6.0, 0.01),
    "kappa-large": lambda: _water(4, 6.0, 6.0, 3.0),
    "wolf": lambda: _water(4, 5.0, 6.2, 0.25, elec="wolf"),
    "argon-half-box": lambda: configs.lj_fcc(ncell=3, rc=2.51, jitter=0.05, seed=4),
    "argon": lambda: configs.lj_fcc(ncell=5, jitter=0.05, seed=4),
    "ghosts": lambda: configs.mixture_box(n_water=40, n_co=30, L=18.0, rc=8.5, water4=True),
    "switched": lambda: configs.mixture_box(n_water=40, n_co=30, L=18.0, rc=8.5, elec="wolf",
                                            switch=True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_exact_pairs_match_oracle(name):
    s = system_of(CASES[name]())
    o = Oracle(s)
    f, t = o.frclong()
    scale = abs(t["uvdw"]) + abs(t["ureal"]) + abs(t["uexcl"]) + abs(t["ufourier"])
    for skin in (0.0, 1.0):
        for wpc in (1, 2, 4, 8):
            print(f"case {name} skin={skin} wpc={wpc}", flush=True)
            eng = Engine(s, precision="fp64")
            eng.set_list_skin(skin / s.params["sigma_base"])
            eng.set_launch_shape(8.0, wpc)
            g, u = eng.frclong()
            eng.close()
            for k in ("n_lj_pairs", "n_elec_pairs", "lj_pair_hash", "elec_pair_hash"):
                assert u[k] == t[k], (k, u[k], t[k])
            assert np.linalg.norm(g - f) <= 1e-12 * np.linalg.norm(f)
            for k in ("uvdw", "ushift", "ureal", "uinter", "virial_inter"):
                assert abs(u[k] - t[k]) <= 1e-12 * max(scale, abs(t[k])), (k, u[k], t[k])
