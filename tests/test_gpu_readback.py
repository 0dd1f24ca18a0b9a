"""Read-backs at sizes around one slot of the pinned ring, between, and where several
threads empty the ring: every value arrives, unchanged."""
import numpy as np
import pytest

from lb_amd import Lattice, abi, make_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,kept", [(abi.STORAGE_F64, np.float64), (abi.STORAGE_F32, np.float32),
                                          (abi.STORAGE_BF16DEV, np.float32)], ids=["f64", "f32", "bf16"])
@pytest.mark.parametrize("n", [(2, 2, 2), (32, 32, 32), (33, 32, 32), (64, 64, 64), (128, 128, 128), (160, 151, 130), (161, 163, 167)], ids=str)
def test_fields_arrive_unchanged(n, storage, kept):
    shape = n[::-1]
    rng = np.random.default_rng(5)
    fields = [1.0 + 0.01 * rng.standard_normal(shape)] + [0.01 * rng.standard_normal(shape) for _ in range(3)]
    L = Lattice(make_desc(np.ones(shape, np.int32), [], storage=storage, arith=abi.ARITH_FAST, periodic=(1, 1, 1),
                          tau=0.6))
    L.init_equilibrium(*fields)
    expect = [f.astype(kept).astype(np.float64) for f in fields]
    for _ in range(2):
        assert all(np.array_equal(a, b) for a, b in zip(L.macroscopic(), expect))
    L.moment_add()
    L.moment_add()
    mean, count = L.moment_avg()
    assert count == 2 and all(np.array_equal(a, b) for a, b in zip(mean, expect))
    assert np.array_equal(L.omega(), np.full(shape, float(kept(1) / kept(0.6))))


def test_populations_arrive_unchanged():
    shape = (64, 64, 80)
    f = np.random.default_rng(6).uniform(0.9, 1.1, (27, *shape))
    L = Lattice(make_desc(np.ones(shape, np.int32), [], storage=abi.STORAGE_F64, arith=abi.ARITH_FAST,
                          periodic=(1, 1, 1), tau=0.6))
    L.set_populations(f)
    assert np.array_equal(L.populations(), f)
    assert np.array_equal(L.population(20), f[20])
