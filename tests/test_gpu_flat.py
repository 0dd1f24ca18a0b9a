"""Periodic boxes whose rows do not fill tiles, with row tiles enough (over 256) that the
step takes 256 consecutive cells a tile, and with one less: every population equals the
oracle's."""
import numpy as np
import pytest

from helpers import OracleLattice, random_velocity_field
from lb_amd import Lattice, abi, make_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(33, 40, 26), (33, 40, 25), (203, 20, 20), (255, 9, 40), (257, 5, 40), (17, 17, 150),
                               (2, 150, 40), (48, 31, 29), (48, 31, 33)], ids=str)
def test_periodic_box_equals_the_oracle(n):
    flags = np.ones(n[::-1], np.int32)
    u = random_velocity_field(flags.shape, 0.05, 3)
    kw = dict(collision=abi.COLLISION_CUM2015, closure=abi.CLOSURE_SMAGORINSKY, storage=abi.STORAGE_F64,
              arith=abi.ARITH_LITERAL, periodic=(1, 1, 1), tau=0.52, c_les=0.1)
    g, o = Lattice(make_desc(flags, [], **kw)), OracleLattice(make_desc(flags, [], **kw))
    for L in (g, o):
        L.init_equilibrium(None, *u)
    for steps in (1, 4):   # both layouts of the state
        for L in (g, o):
            L.step(steps)
        assert np.array_equal(g.populations(), o.populations())
    mass = g.step_diagnostics()[0]   # of the state before the step, summed in FP64
    assert abs(mass - o.populations().sum()) < 1e-9 * flags.size
