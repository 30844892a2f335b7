"""The list build's launch shapes: binning workgroups of 256 and 1024 threads
(up to 2,048 cells and above) and placing workgroups of 64 to 1024 threads (by
atoms per column), from the cells a system is given; the pairs found are the
oracle's, exactly, on a first build and on a rebuild after every atom moved."""
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
