"""The diagnostics step that allocates nothing takes a lattice with boundaries whose
rows fill seven 64-wide tiles and two 256-wide ones: 231 868 tiles of 256 cells, less
than its array holds, where two wide tiles a row would make 264 992."""
import numpy as np
import pytest

from lb_amd import Lattice, abi, make_desc

pytestmark = pytest.mark.gpu


def test_tile_width_leaves_the_lattice_within_the_array():
    n = (410, 364, 364)
    flags = np.ones(n[::-1], np.int32)
    flags[5, 5, 5] = 0
    L = Lattice(make_desc(flags, [], storage=abi.STORAGE_F16DEV, arith=abi.ARITH_FAST, periodic=(1, 1, 1), tau=0.6))
    L.init_equilibrium()
    mass, j, _ = L.step_diagnostics_noalloc()
    cells = flags.size - 1
    assert abs(mass / cells - 1) < 1e-5 and np.abs(j).max() < 1e-3   # at rest, FP32 sums of 27 weights
    L.close()
