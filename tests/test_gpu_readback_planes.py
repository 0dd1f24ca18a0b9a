"""Read-backs of some of the planes, and of planes into shared memory, at sizes that one
pinned slot holds, between, and where several threads empty the ring: a plane that is
not wanted is left out, and of planes into one array the last one's values stay."""
import ctypes

import numpy as np
import pytest

from lb_amd import Lattice, abi, make_desc

pytestmark = pytest.mark.gpu

SIZES = [(20, 20, 20), (32, 32, 33), (90, 80, 70), (234, 233, 233)]


def lattice(n):
    shape = n[::-1]
    # values that 16-bit storage keeps no better than the four planes differ from one another
    u = [np.full(shape, v) + 1e-3 * (np.arange(n[0]) % 7) for v in (0.01, 0.02, 0.03)]
    L = Lattice(make_desc(np.ones(shape, np.int32), [], storage=abi.STORAGE_F16DEV, arith=abi.ARITH_FAST,
                          periodic=(1, 1, 1), tau=0.6))
    L.init_equilibrium(None, *u)
    return L


def read(L, arrays):
    none = ctypes.cast(None, ctypes.POINTER(ctypes.c_double))
    st = L._lib.lbm_get_macroscopic(L._h, *[none if a is None else abi.ptr(a) for a in arrays])
    assert st == abi.LBM_OK


@pytest.mark.parametrize("n", SIZES, ids=str)
def test_wanted_planes_alone(n):
    L = lattice(n)
    full = [np.empty(n[::-1]) for _ in range(4)]
    read(L, full)
    assert not np.array_equal(full[1], full[2]) and not np.array_equal(full[2], full[3])
    for wanted in ([0, 2], [1, 3], [3], [0, 1, 3], []):
        some = [np.full(n[::-1], -7.0) if k in wanted else None for k in range(4)]
        read(L, some)
        for k in wanted:
            assert np.array_equal(some[k], full[k])
    L.close()


@pytest.mark.parametrize("n", SIZES, ids=str)
def test_planes_in_shared_memory(n):
    L = lattice(n)
    full = [np.empty(n[::-1]) for _ in range(4)]
    read(L, full)
    a, b = np.empty(n[::-1]), np.empty(n[::-1])
    for order in ([a, b, a, b], [a, a, a, a], [a, None, b, a]):
        read(L, order)
        for x in (a, b):
            last = [k for k in range(4) if order[k] is x]
            assert not last or np.array_equal(x, full[last[-1]])
    both = np.empty(2 * a.size)   # uy's second half is uz's first
    half = a.size // 2
    read(L, [None, None, both[:a.size], both[half:half + a.size]])
    assert np.array_equal(both[:half], full[2].ravel()[:half])
    assert np.array_equal(both[half:half + a.size], full[3].ravel())
    L.close()


def test_lattices_of_several_threads_share_the_pinned_blocks():
    import threading
    for _ in range(2):   # the second round starts without a context: the blocks were given back
        bad = []

        def work(k):
            L = Lattice(make_desc(np.ones((16, 20, 24), np.int32), [], storage=abi.STORAGE_F64, arith=abi.ARITH_FAST,
                                  periodic=(1, 1, 1), tau=0.6))
            rho = 1.0 + 0.01 * (k + np.random.default_rng(k).random((16, 20, 24)))
            L.init_equilibrium(rho, None, None, None)
            for _ in range(40):
                if not np.array_equal(L.macroscopic()[0], rho):
                    bad.append(k)
            L.close()

        team = [threading.Thread(target=work, args=(k,)) for k in range(6)]
        for t in team:
            t.start()
        for t in team:
            t.join()
        assert not bad
