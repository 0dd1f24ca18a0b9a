"""Diagnostics of a step that takes its tiles from the last to the first, or with the
row groups of a plane rotated: mass and momentum equal the sums over the state that
the step collides, so that no tile's record is lost, doubled or overwritten.  Rows off
the cache lines with walls, and larger than the cache: a start shifted in z gives the
shifted state, bit for bit."""
import numpy as np
import pytest

from helpers import random_velocity_field
from lb_amd import Lattice, abi, make_desc

pytestmark = pytest.mark.gpu


def start(n, walls):
    shape = n[::-1]
    flags = np.ones(shape, np.int32)
    if walls:
        flags[:, 0] = flags[:, -1] = 0
    u = [np.tile(c, (-(-shape[0] // 8), -(-shape[1] // 8), -(-shape[2] // 8)))[:shape[0], :shape[1], :shape[2]]
         for c in random_velocity_field((8, 8, 8), 0.02, 5)]
    return flags, [np.where(flags == 0, 0.0, c + 0.002 * (1 + np.arange(shape[0])).reshape(-1, 1, 1) / shape[0]) for c in u]


CASES = [((160, 160, 160), abi.STORAGE_F32, False), ((203, 160, 131), abi.STORAGE_F32, False),
         ((192, 192, 160), abi.STORAGE_BF16DEV, False), ((203, 130, 110), abi.STORAGE_F32, True),
         ((203, 130, 200), abi.STORAGE_F16DEV, True), ((150, 100, 90), abi.STORAGE_F64, True),
         ((192, 130, 110), abi.STORAGE_F32, True), ((256, 34, 300), abi.STORAGE_F16DEV, True)]


@pytest.mark.parametrize("n,storage,walls", CASES, ids=str)
def test_diagnostics_are_the_sums_of_the_state(n, storage, walls):
    flags, u = start(n, walls)
    L = Lattice(make_desc(flags, [], storage=storage, arith=abi.ARITH_FAST, periodic=(1, 0 if walls else 1, 1), tau=0.55))
    L.init_equilibrium(None, *u)
    cells = int((flags != 0).sum())
    for _ in range(4):   # both parities
        sums = np.asarray(L.conservation(), dtype=float)
        mass, j, _ = L.step_diagnostics()
        # FP32 cell values of 1 and 0.02 within some 1e-7; a tile is 256 cells of at most 6e6
        assert abs(mass - sums[0]) < 1e-6 * cells
        assert np.abs(j - sums[1:4]).max() < 1e-6 * 0.02 * cells
    L.close()


@pytest.mark.parametrize("n,storage,walls", [c for c in CASES if c[2]], ids=str)
def test_walled_lattices_are_shift_invariant(n, storage, walls):
    flags, u = start(n, walls)
    out = []
    for f in (u, [np.roll(c, 3, 0) for c in u]):
        L = Lattice(make_desc(flags, [], closure=abi.CLOSURE_SMAGORINSKY, storage=storage, arith=abi.ARITH_FAST,
                              periodic=(1, 0, 1), tau=0.55, c_les=0.1))
        L.init_equilibrium(None, *f)
        L.step(5)
        out.append(L.macroscopic())
        L.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(np.roll(a, 3, 0), b)
