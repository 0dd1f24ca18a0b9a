"""The random bits of stochastic rounding belong to a cell's place in the caller's
lattice, not to the layout that the core chooses: away from walls, a lattice
without index wrap draws what a periodic box draws whose rows hold a cache line of
64 cells before the lattice's own, and whose other axes hold one cell around it."""
import numpy as np
import pytest

from lb_amd import Lattice, abi, make_desc

pytestmark = pytest.mark.gpu

LINE = 64   # 16-bit populations in a cache line


@pytest.mark.parametrize("storage", [abi.STORAGE_F16DEV_SR, abi.STORAGE_BF16DEV_SR], ids=["f16sr", "bf16sr"])
@pytest.mark.parametrize("n,left,periodic", [
    ((10, 9, 8), 0, (0, 0, 0)), ((10, 9, 8), 2, (0, 0, 0)), ((62, 9, 8), 0, (0, 1, 1)), ((63, 9, 8), 1, (0, 0, 1)),
    ((64, 9, 8), 0, (0, 1, 0)), ((130, 10, 9), 65, (0, 0, 0)), ((33, 9, 8), 0, (1, 0, 1))], ids=str)
def test_bits_do_not_depend_on_the_layout(n, left, periodic, storage):
    nx, ny, nz = n
    lead = (0 if periodic[0] else LINE, 0 if periodic[1] else 1, 0 if periodic[2] else 1)
    box = (nx if periodic[0] else -(-(LINE + nx + 1) // LINE) * LINE, ny + 2 * lead[1], nz + 2 * lead[2])
    flags = np.ones((nz, ny, nx), np.int32)
    flags[:, :, :left] = 0
    kw = dict(storage=storage, arith=abi.ARITH_FAST, closure=abi.CLOSURE_NONE, tau=0.6)
    a = Lattice(make_desc(flags, [], periodic=periodic, **kw))
    b = Lattice(make_desc(np.ones(box[::-1], np.int32), [], periodic=(1, 1, 1), **kw))
    for L in (a, b):   # one density everywhere, between two values of the format
        L.init_equilibrium(np.full(flags.shape if L is a else box[::-1], 1.0037), None, None, None)
    keep = [slice(None)] * 3
    for k, steps in enumerate((1, 1, 1)):
        for L in (a, b):
            L.step(steps)
        for i in range(3):   # no wall within the steps taken
            if not periodic[i]:
                keep[i] = slice((left if i == 0 else 0) + k + 1, n[i] - k - 1)
        z, y, x = keep[::-1]
        fa = a.populations()
        fb = b.populations()[:, lead[2]:lead[2] + nz, lead[1]:lead[1] + ny, lead[0]:lead[0] + nx]
        assert fa[:, z, y, x].size and len(np.unique(fa[1, z, y, x])) > 1
        assert np.array_equal(fa[:, z, y, x], fb[:, z, y, x])
