"""Row pitches around 15, 17 and 20 cache lines (16 FP64 populations each), which take a
line more: every population equals the oracle's, also where the last row's overhang
decides the size of a plane."""
import numpy as np
import pytest

from helpers import OracleLattice, random_velocity_field
from lb_amd import Lattice, abi, make_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("left,right", [(0, 0), (3, 1)], ids=str)
@pytest.mark.parametrize("nx", [222, 223, 238, 239, 254, 255, 270, 271, 302, 318])
def test_long_rows_equal_the_oracle(nx, left, right):
    flags = np.zeros((3, 4, left + nx + right), np.int32)
    flags[:, :, left:left + nx] = 1
    u = [c[:3, :4, :flags.shape[2]].copy() for c in random_velocity_field((4, 4, 512), 0.03, 8)]
    kw = dict(collision=abi.COLLISION_CUM2015, storage=abi.STORAGE_F64, arith=abi.ARITH_LITERAL, periodic=(0, 0, 1),
              tau=0.6)
    g, o = Lattice(make_desc(flags, [], **kw)), OracleLattice(make_desc(flags, [], **kw))
    for L in (g, o):
        L.init_equilibrium(None, *u)
    for steps in (1, 2):
        for L in (g, o):
            L.step(steps)
        assert np.array_equal(g.populations()[:, flags != 0], o.populations()[:, flags != 0])
