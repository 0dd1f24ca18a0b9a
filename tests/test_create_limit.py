"""Lattices beyond the 32-bit plane offsets are refused before the flag grid is read:
its memory allows no access here, so that a read ends the child process."""
import subprocess
import sys

import pytest

CHILD = """
import ctypes, sys
import numpy as np
from lb_amd import abi, make_desc
libc = ctypes.CDLL(None, use_errno=True)
libc.mmap.restype = ctypes.c_void_p
libc.mmap.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_long]
page = libc.mmap(None, 4096, 0, 0x22, -1, 0)   # PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS
assert page not in (None, ctypes.c_void_p(-1).value)
n, storage, periodic = eval(sys.argv[1])
d = make_desc(np.ones((2, 2, 2), np.int32), [], tau=0.6, storage=storage, arith=abi.ARITH_FAST, periodic=periodic)
d.nx, d.ny, d.nz = n
d.flags = ctypes.cast(page, type(d.flags))
h = ctypes.c_void_p()
print("status", abi.load_core().lbm_create(ctypes.byref(d), ctypes.byref(h)), abi.LBM_E_ARG)
"""


@pytest.mark.parametrize("n,storage,periodic", [
    ((4096, 4096, 4096), 0, (1, 1, 1)), ((4096, 4096, 4096), 2, (0, 0, 0)), ((1, 2 ** 31 - 1, 2 ** 31 - 1), 1, (0, 0, 0)),
    ((2 ** 31 - 1, 2 ** 31 - 1, 2 ** 31 - 1), 0, (0, 0, 0)), ((1024, 1024, 512), 0, (1, 1, 1)),
    ((1024, 1024, 510), 0, (0, 0, 0))], ids=str)
def test_refused_without_reading_the_flags(n, storage, periodic):
    r = subprocess.run([sys.executable, "-c", CHILD, repr((n, storage, periodic))], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr[-500:]
    _, status, expect = r.stdout.split()
    assert status == expect
