"""Row pitch and halo along x without index wrap, at the widths where the last
cell, the halo and the next row's halo meet the ends of cache lines (16 FP64
populations): every population equals the oracle's."""
import numpy as np
import pytest

from helpers import OracleLattice, random_velocity_field
from lb_amd import Lattice, abi, make_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("left,right", [(0, 0), (1, 1), (0, 3), (2, 0), (16, 0), (17, 2), (32, 0)], ids=str)
@pytest.mark.parametrize("nx", [1, 13, 14, 15, 16, 17, 32])
@pytest.mark.parametrize("periodic", [(0, 1, 1), (0, 0, 1), (0, 0, 0)], ids=str)
def test_rows_without_wrap_equal_the_oracle(nx, left, right, periodic):
    flags = np.zeros((4, 5, left + nx + right), np.int32)
    flags[:, :, left:left + nx] = 1
    u = random_velocity_field((4, 8, 64), 0.03, 7)
    u = [np.ascontiguousarray(c[:4, :5, :flags.shape[2]]) for c in u]
    kw = dict(collision=abi.COLLISION_CUM2015, storage=abi.STORAGE_F64, arith=abi.ARITH_LITERAL, periodic=periodic,
              tau=0.6)
    g, o = Lattice(make_desc(flags, [], **kw)), OracleLattice(make_desc(flags, [], **kw))
    for L in (g, o):
        L.init_equilibrium(None, *u)
    fluid = flags != 0
    for steps in (1, 2):   # both layouts of the state
        for L in (g, o):
            L.step(steps)
        assert np.array_equal(g.populations()[:, fluid], o.populations()[:, fluid])
