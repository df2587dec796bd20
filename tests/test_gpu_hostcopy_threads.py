"""GPU test of the field copies where they have two and three helper threads
(24 and 32 MiB of host values, n = 147 and 162 on), which test_gpu_hostcopy.py
stops short of: bit-exact round trips in every storage type, also right after
an OpenMP region, whose threads still hold the CPUs when the helpers start, and
from a pinned buffer."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
import pyetd
from conftest import small_params

pytestmark = pytest.mark.gpu


def values(n):
    r = np.random.default_rng(n)
    a = r.uniform(-1, 1, n ** 3) * 10.0 ** r.integers(-30, 30, n ** 3)
    a[:4] = np.inf, -np.inf, np.nan, -0.0
    return a


def check(L, g, a, buf, before, precision):
    """Set a, read into buf, each after before()."""
    p = [x.ctypes.data_as(C.POINTER(C.c_double)) for x in (a, buf)]
    buf[:] = 7.0
    before()
    assert L.etd_set_field(g.ctx, 0, p[0]) == 0
    before()
    assert L.etd_get_field(g.ctx, 0, p[1]) == 0
    with np.errstate(over="ignore"):
        want = a if precision == 0 else a.astype(np.float32).astype(np.float64)
    assert np.array_equal(buf.view(np.uint64), want.copy().view(np.uint64))


@pytest.fixture
def pinned():
    """pinned(count): an array in memory that the runtime pinned."""
    L, got = pyetd.lib(), []

    def alloc(count):
        p = C.c_void_p()
        assert L.hipHostMalloc(C.byref(p), C.c_size_t(8 * count), C.c_uint(0)) == 0
        got.append(p)
        return np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (count,))

    yield alloc
    for p in got:
        assert L.hipHostFree(p) == 0


@pytest.fixture(scope="module")
def openmp():
    """A parallel region of the oracle's (a ghost fill and a step of a small box)."""
    o = O.Oracle(small_params(n=20, nac=1))
    o.set_field(0, np.zeros((20, 20, 20)))
    return lambda: o.step(1)


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("n", [144, 148, 160, 164, 196])
def test_round_trip(n, precision, pinned, openmp):
    L = pyetd.lib()
    g = pyetd.Etd.from_dict(dict(small_params(n=n, nac=1), precision=precision))
    a, b = values(n), np.empty(n ** 3)
    for before in (lambda: None, openmp):
        for _ in range(3):
            print(f"round trip n={n} precision={precision}", flush=True)
            check(L, g, a, b, before, precision)
    pa, pb = pinned(n ** 3), pinned(n ** 3)
    pa[:] = a
    print(f"pinned n={n} precision={precision}", flush=True)
    check(L, g, pa, pb, lambda: None, precision)
    check(L, g, a, pb, openmp, precision)
    g.close()
