"""Tiles of the step: runs of consecutive cells on periodic lattices whose rows
do not fill tiles, and the box of non-solid cells elsewhere, at the sizes where
rows, planes and tiles end inside one another."""
import numpy as np
import pytest

from helpers import OracleLattice, cavity_setup, random_velocity_field
from lb_amd import Lattice, abi, make_desc

pytestmark = pytest.mark.gpu

BOXES = [(2, 2, 2), (7, 5, 3), (33, 18, 4), (63, 4, 5), (203, 9, 5), (255, 2, 3), (256, 3, 2), (257, 3, 2)]


@pytest.mark.parametrize("n", BOXES, ids=str)
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


@pytest.mark.parametrize("storage", [abi.STORAGE_F32, abi.STORAGE_F16DEV, abi.STORAGE_BF16DEV], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("n", BOXES, ids=str)
def test_periodic_box_is_shift_invariant(n, storage):
    flags = np.ones(n[::-1], np.int32)
    u = random_velocity_field(flags.shape, 0.05, 4)
    shift = (1, 1, n[0] // 2 + 1)
    out = []
    for f in (u, [np.roll(c, shift, (0, 1, 2)) for c in u]):
        L = Lattice(make_desc(flags, [], closure=abi.CLOSURE_SMAGORINSKY, storage=storage, arith=abi.ARITH_FAST,
                              periodic=(1, 1, 1), tau=0.52, c_les=0.1))
        L.init_equilibrium(None, *f)
        L.step(5)
        out.append(L.macroscopic())
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(np.roll(a, shift, (0, 1, 2)), b)


@pytest.mark.parametrize("margin", [(0, 0, 0), (1, 2, 3), (40, 0, 1), (64, 1, 0)], ids=str)
@pytest.mark.parametrize("n", [6, 33])
def test_cavity_inside_solid_margins_equals_the_oracle(n, margin):
    f0, bc, u0 = cavity_setup(n)
    mx, my, mz = margin
    pad = ((mz, 1), (my, 2), (mx, 3))
    flags, ux = np.pad(f0, pad), np.pad(u0, pad)
    for b in bc:
        b.x, b.y, b.z = b.x + mx, b.y + my, b.z + mz
    kw = dict(collision=abi.COLLISION_CUM2015, storage=abi.STORAGE_F64, arith=abi.ARITH_LITERAL, tau=0.524)
    g, o = Lattice(make_desc(flags, bc, **kw)), OracleLattice(make_desc(flags, bc, **kw))
    for L in (g, o):
        L.init_equilibrium(None, ux, None, None)
    for steps in (1, 4):
        for L in (g, o):
            L.step(steps)
        assert np.array_equal(g.populations(), o.populations())


def test_all_solid_lattice_runs():
    L = Lattice(make_desc(np.zeros((3, 4, 5), np.int32), [], storage=abi.STORAGE_F32, arith=abi.ARITH_FAST))
    L.init_equilibrium()
    L.step(3)
    assert all(not m.any() for m in L.macroscopic())
