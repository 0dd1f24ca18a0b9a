"""Lattices with walls in y whose row groups the step hands to the XCDs in another
order in every plane, with a lid and without: row groups a plane around eight and
even, a last group partly filled, more planes than eight.  Every population equals
the oracle's."""
import numpy as np
import pytest

from helpers import OracleLattice, random_velocity_field
from lb_amd import Lattice, abi, host, make_desc

pytestmark = pytest.mark.gpu


def lid(n):
    g = np.zeros(n[::-1], np.int32)
    g[1:-1, 1:-1, 1:-1] = 1
    m = host.Mesher(g, 1.0, 1.0, (0.0, 0.0, 0.0))
    m.wall()
    top, big = n[1] - 2, 1e4
    m.inlet((-big, top - 0.75, -big), (big, top - 0.25, big), (-big, top - 0.75, big), -1, (0.0, 1.0, 0.0),
            (0.05, 0.0, 0.0), abi.BC_INLET_MOVING_WALL)
    return m.compile()


# the box's rows (n - 2) in groups of 8, 4, 2 and 1; sizes on both sides of the rule's line
@pytest.mark.parametrize("n", [(34, 66, 162), (66, 34, 170), (66, 39, 150), (130, 18, 140), (130, 22, 118), (258, 10, 130),
                               (66, 30, 40), (130, 18, 160), (130, 22, 140), (258, 10, 160)], ids=str)
def test_lid_cavity_equals_the_oracle(n):
    flags, bc = lid(n)
    ux = np.where(flags == -1, 0.05, 0.0)
    kw = dict(collision=abi.COLLISION_CUM2015, storage=abi.STORAGE_F64, arith=abi.ARITH_LITERAL, tau=0.524)
    g, o = Lattice(make_desc(flags, bc, **kw)), OracleLattice(make_desc(flags, bc, **kw))
    for L in (g, o):
        L.init_equilibrium(None, ux, None, None)
    for steps in (1, 2):   # both layouts of the state
        for L in (g, o):
            L.step(steps)
        assert np.array_equal(g.populations(), o.populations())


@pytest.mark.parametrize("n", [(64, 34, 162), (128, 18, 160), (256, 10, 160)], ids=str)
def test_channel_equals_the_oracle(n):
    flags = np.ones(n[::-1], np.int32)
    flags[:, 0] = flags[:, -1] = 0
    u = [np.where(flags == 0, 0.0, np.tile(c, (-(-n[2] // 8), 1, n[0] // 8))[:n[2]])
         for c in random_velocity_field((8, n[1], 8), 0.03, 6)]
    kw = dict(collision=abi.COLLISION_CUM2015, storage=abi.STORAGE_F64, arith=abi.ARITH_LITERAL, tau=0.55,
              periodic=(1, 0, 1))
    g, o = Lattice(make_desc(flags, [], **kw)), OracleLattice(make_desc(flags, [], **kw))
    for L in (g, o):
        L.init_equilibrium(None, *u)
    for steps in (1, 2):
        for L in (g, o):
            L.step(steps)
        assert np.array_equal(g.populations(), o.populations())
