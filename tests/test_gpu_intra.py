"""The intramolecular pair terms by one wave per term (k_intra_tw) for
molecules of up to three, four and six sites and terms, at the edges of its
workgroups (64 molecules), on the stream of the reciprocal forces and on the
main one, with ghosts, and with molecules longer than half the box (1-2, 1-3
and 1-4 pairs that then take their images); larger molecules and the adjoint
by one thread per molecule.  FP64 against the oracle: forces within 1e-12 of
the norm, energies within 1e-12 of the pair energies' scale (sums of at most
1e5 terms of a few 1e-16 each)."""
import numpy as np
import pytest

from mspms2_amd import configs
from mspms2_amd.engine import Engine
from oracle.oracle import Oracle
from tests.test_gpu_nvt_solve import _chain, _water
from tests.util import system_of

pytestmark = pytest.mark.gpu


def _stretched(rd, seed, factor):
    """Molecules scattered over the box: sites apart by more than half of it."""
    s = system_of(rd)
    rng = np.random.default_rng(seed)
    L = s.params["boxlx"]
    for a in (s.xx, s.yy, s.zz):
        a += factor * L * rng.uniform(-1.0, 1.0, a.shape)
    return s


CASES = {
    "water-1": lambda: system_of(_water(1)),
    "water-64": lambda: system_of(_water(64)),
    "water-65": lambda: system_of(_water(65)),
    "water-wolf": lambda: system_of(configs.water_box(n_side=4, L=12.4, rc=5.0, kappa=0.25,
                                                      kmax=2, ksqmax=4, elec="wolf", seed=3)),
    "chain-65": lambda: system_of(_chain(65)),
    "butane-64": lambda: system_of(configs.butane_box(nmol=64)),
    "zoo-43": lambda: system_of(configs.bonded_zoo(nmole=43)),
    "ghosts": lambda: system_of(configs.mixture_box(n_water=40, n_co=30, L=18.0, rc=8.5,
                                                    water4=True)),
    "water-long": lambda: _stretched(_water(65), 1, 0.4),
    "chain-long": lambda: _stretched(_chain(65), 2, 0.4),
    "butane-long": lambda: _stretched(configs.butane_box(nmol=64), 3, 0.4),
}


@pytest.mark.parametrize("name", list(CASES))
def test_intramolecular_terms_match_oracle(name):
    s = CASES[name]()
    f, t = Oracle(s).frclong()
    scale = sum(abs(t[k]) for k in ("uvdw", "ureal", "uexcl", "ufourier"))
    print(f"case {name}", flush=True)
    eng = Engine(s, precision="fp64")
    g, u = eng.frclong()
    eng.close()
    assert np.linalg.norm(g - f) <= 1e-12 * np.linalg.norm(f)
    for k in ("uvdw", "ureal", "uexcl", "virial_inter"):
        assert abs(u[k] - t[k]) <= 1e-12 * max(scale, abs(t[k])), (k, u[k], t[k])
