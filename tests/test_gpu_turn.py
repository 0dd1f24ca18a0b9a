"""Lattices larger than the cache in front of the HBM, where odd steps take the
tiles from the last to the first and either parity may take the streaming hint:
a shifted start gives the shifted state, bit for bit, and the diagnostics of a
step do not depend on its parity's tile order."""
import numpy as np
import pytest

from helpers import random_velocity_field
from lb_amd import Lattice, abi, make_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,storage,wall", [
    ((203, 160, 131), abi.STORAGE_F32, False),    # rows off the cache lines
    ((150, 150, 113), abi.STORAGE_F32, False),    # the same, little larger than the cache
    ((160, 160, 160), abi.STORAGE_F32, False),
    ((192, 160, 161), abi.STORAGE_F32, False),
    ((192, 192, 160), abi.STORAGE_BF16DEV, False),
    ((144, 112, 112), abi.STORAGE_F64, False),
    ((160, 130, 130), abi.STORAGE_F32, True),
    ((190, 160, 130), abi.STORAGE_F32, True),
    ((222, 170, 150), abi.STORAGE_F16DEV, True),
], ids=str)
def test_large_lattices_are_shift_invariant(n, storage, wall):
    shape = n[::-1]
    flags = np.ones(shape, np.int32)
    if wall:
        flags[:, :, 0] = 0
    u = [np.tile(c, (-(-shape[0] // 8), -(-shape[1] // 8), -(-shape[2] // 8)))[:shape[0], :shape[1], :shape[2]]
         for c in random_velocity_field((8, 8, 8), 0.02, 5)]
    u = [np.where(flags == 0, 0.0, c + 0.001 * np.arange(shape[0]).reshape(-1, 1, 1) / shape[0]) for c in u]
    shift = (3, 1)
    out = []
    for f in (u, [np.roll(c, shift, (0, 1)) for c in u]):
        L = Lattice(make_desc(flags, [], closure=abi.CLOSURE_SMAGORINSKY, storage=storage, arith=abi.ARITH_FAST,
                              periodic=(0 if wall else 1, 1, 1), tau=0.55, c_les=0.1))
        L.init_equilibrium(None, *f)
        L.step(3)
        mass = [L.step_diagnostics()[0], L.step_diagnostics()[0]]
        out.append(L.macroscopic() + [mass])
        L.close()
    for a, b in zip(out[0][:4], out[1][:4]):
        assert np.isfinite(a).all() and np.array_equal(np.roll(a, shift, (0, 1)), b)
    cells = int((flags != 0).sum())
    assert np.allclose(out[0][4] + out[1][4], cells, rtol=2e-3)
