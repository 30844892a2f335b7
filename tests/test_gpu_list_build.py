"""The list build's launch shapes: binning workgroups of 256 and 1024 threads
(up to 2,048 cells and above) and placing workgroups of 64 to 1024 threads (by
atoms per column), from the cells a system is given; the pairs found are the
oracle's, exactly.  And the build of up to 1,024 atoms by one workgroup, on a
first build, on reuse of the list and on a rebuild."""
import numpy as np
import pytest

from mspms2_amd import configs
from mspms2_amd.engine import Engine
from oracle.oracle import Oracle
from tests.util import system_of

pytestmark = pytest.mark.gpu


# atoms per cell: 6,912 atoms in 3,375 cells of 225 columns, in 2,197 of 169, in
# 1,728 of 144, in 729 of 81, and in 64 of 16 (columns of 432: 1024 threads)
@pytest.mark.parametrize("cell_atoms", [2.0, 3.0, 3.3, 8.0, 64.0])
def test_pairs_of_every_launch_shape(cell_atoms):
    s = system_of(configs.lj_fcc(ncell=12, jitter=0.05, seed=4))
    f, t = Oracle(s).frclong()
    print(f"atoms per cell {cell_atoms}", flush=True)
    eng = Engine(s, precision="fp64")
    eng.set_launch_shape(cell_atoms, 4)
    for _ in range(2):
        g, u = eng.frclong()
        for k in ("n_lj_pairs", "lj_pair_hash"):
            assert u[k] == t[k], (k, u[k], t[k])
        assert np.linalg.norm(g - f) <= 1e-12 * np.linalg.norm(f)
    eng.close()


SMALL = {
    "water-1": lambda: [configs.water_box(n_side=1, L=8.0, rc=3.9, kappa=0.5, nmol=1, seed=2)],
    "water-341": lambda: [configs.water_box(n_side=7, L=21.7, rc=7.0, nmol=341, seed=2)],  # 1,023
    "water-342": lambda: [configs.water_box(n_side=7, L=21.7, rc=7.0, nmol=342, seed=2)],  # 1,026
    "batch": lambda: [configs.water_box(n_side=5, L=15.5, rc=7.0, nmol=n, seed=n)
                      for n in (1, 125, 30)],
    "ghosts": lambda: [configs.mixture_box(n_water=40, n_co=30, L=18.0, rc=8.5, water4=True)],
}


@pytest.mark.parametrize("name", list(SMALL))
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_pairs_of_small_systems(name, precision):
    systems = [system_of(rd) for rd in SMALL[name]()]
    print(f"{name} {precision}", flush=True)
    eng = Engine.replicas(systems, precision=precision)
    skin = 0.6 / systems[0].params["sigma_base"]
    eng.set_list_skin(skin)
    rng = np.random.default_rng(5)
    # from the first positions: none, every atom by less than half the skin
    # (reuse), by more (rebuild)
    unit = [rng.uniform(-1.0, 1.0, (3, s.natom)) / np.sqrt(3.0) for s in systems]
    for d in (0.0, 0.45 * skin, 0.9 * skin):
        xs = [np.stack([s.xx, s.yy, s.zz]) + d * u for s, u in zip(systems, unit)]
        g, terms = eng.frclong(*eng.pack(xs))
        terms = [terms] if isinstance(terms, dict) else terms
        for s, x, f, u in zip(systems, xs, eng.unpack(g), terms):
            fo, to = Oracle(s).frclong(*x)
            if precision == "fp64":
                for k in ("n_lj_pairs", "n_elec_pairs", "lj_pair_hash", "elec_pair_hash"):
                    assert u[k] == to[k], (k, u[k], to[k])
            # FP32 pair terms of the mixed kernel: 6e-8 each, with cancellation
            tol = 1e-12 if precision == "fp64" else 2e-5
            assert np.linalg.norm(f - fo) <= tol * np.linalg.norm(fo)
    eng.close()


# with a skin, several passes of the cell scan: more than 8,192 cells by 1024
# threads, and, beside the Ewald kernels, more than 4,096 by 256
SKINNED = {
    "lj-19652": lambda: configs.lj_fcc(ncell=17, jitter=0.05, seed=4),
    "water-3375": lambda: configs.water_box(n_side=15, L=46.56, rc=8.0, kappa=0.35, kmax=3,
                                            ksqmax=9, seed=4),
}


@pytest.mark.parametrize("name", list(SKINNED))
def test_pairs_of_large_grids_with_a_skin(name):
    s = system_of(SKINNED[name]())
    print(f"{name} natom={s.natom}", flush=True)
    eng = Engine(s, precision="fp64")
    skin = (0.6 if name.startswith("water") else 0.2) / (
        s.params["sigma_base"] if name.startswith("water") else 1.0)
    eng.set_list_skin(skin)
    eng.set_launch_shape(2.0, 4)
    x = np.stack([s.xx, s.yy, s.zz])
    u = np.random.default_rng(5).uniform(-1.0, 1.0, x.shape) / np.sqrt(3.0)
    # a first build, a step that reuses the list, a rebuild
    for d, builds in ((0.0, 1), (0.45 * skin, 1), (0.9 * skin, 2)):
        g, t = eng.frclong(*(x + d * u))
        assert eng.list_builds() == builds
        f, to = Oracle(s).frclong(*(x + d * u))
        for k in ("n_lj_pairs", "n_elec_pairs", "lj_pair_hash", "elec_pair_hash"):
            assert t[k] == to[k], (d, k, t[k], to[k])
        assert np.linalg.norm(g - f) <= 1e-12 * np.linalg.norm(f)
    eng.close()


@pytest.mark.parametrize("nmol", [125, 512])     # built in one launch, and in five
def test_half_and_full_lists_in_turn(nmol):
    """The mixed kernel's half lists, whose reuse leaves the exact kernel's
    positions as they were, and the adjoint's full lists on one engine: each
    after moves of less than half the skin, forces against the oracle."""
    s = system_of(configs.water_box(n_side=8, L=24.9, rc=8.0, kappa=0.35, kmax=3, ksqmax=9,
                                    nmol=nmol, seed=4))
    print(f"half and full lists {s.natom}", flush=True)
    eng = Engine(s, precision="mixed")
    skin = 1.0 / s.params["sigma_base"]
    eng.set_list_skin(skin)
    x = np.stack([s.xx, s.yy, s.zz])
    u = np.random.default_rng(5).uniform(-1.0, 1.0, x.shape) / np.sqrt(3.0)
    for k, exact in enumerate([False, False, True, True, False, False, True]):
        xk = x + 0.07 * k * skin * u
        g = eng.param_grad(*xk)[0] if exact else eng.frclong(*xk)[0]
        f, _ = Oracle(s).frclong(*xk)
        assert np.linalg.norm(g - f) <= (1e-12 if exact else 2e-5) * np.linalg.norm(f), (k, exact)
    eng.close()
