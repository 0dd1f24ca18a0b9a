"""Equilibrium inlet and interpolated outlet where they run after the step
(ghost layers along z), 32 lanes a node: node counts around a workgroup's eight,
irregular nodes among them.  Every population equals the oracle's."""
import numpy as np
import pytest

from helpers import OracleLattice, bc_nodes
from lb_amd import Lattice, abi, make_desc
from oracle import mesher_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [abi.STORAGE_F64, abi.STORAGE_F32], ids=["f64", "f32"])
@pytest.mark.parametrize("ny,nz", [(3, 3), (4, 4), (6, 5), (9, 6), (12, 11)])
def test_inlet_and_outlet_equal_the_oracle(ny, nz, storage):
    flags, bc = mo.channel(8, ny, nz)
    solid = flags == 0
    ux = np.where(solid, 0.0, 0.04 + 0.005 * np.random.default_rng(3).standard_normal(flags.shape))
    kw = dict(collision=abi.COLLISION_CUM2015, storage=storage, arith=abi.ARITH_LITERAL, tau=0.53, nu=0.01,
              compat=abi.COMPAT_REFERENCE)
    g, o = (L(make_desc(flags, bc_nodes(bc), **kw)) for L in (Lattice, OracleLattice))
    for L in (g, o):
        L.init_equilibrium(None, ux, None, None)
    for steps in (1, 4):
        for L in (g, o):
            L.step(steps)
        assert np.array_equal(g.populations()[:, ~solid], o.populations()[:, ~solid])
