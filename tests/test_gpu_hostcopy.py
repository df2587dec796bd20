"""GPU test of the field copies between host and device: every size at which
the copy changes its way (direct, two chunks on the calling thread, chunks
shared by threads, a last chunk that is short), in both storage types, from
buffers at any alignment.  What is read back is what was set, to the bit
(FP32 storage: what a cast gives)."""
import ctypes as C

import numpy as np
import pytest

import pyetd
from conftest import small_params

pytestmark = pytest.mark.gpu


def at(offset, count):
    """count doubles that start offset bytes past a 64-byte boundary."""
    raw = np.empty(8 * count + 128, np.uint8)
    lead = -raw.ctypes.data % 64 + offset
    return raw[lead: lead + 8 * count].view(np.float64)


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("n", [12, 48, 52, 80, 84, 100, 104, 128, 132])
def test_field_round_trip(n, precision):
    print(f"round trip n={n} precision={precision}", flush=True)
    L = pyetd.lib()
    g = pyetd.Etd.from_dict(dict(small_params(n=n, nac=2), precision=precision))
    r = np.random.default_rng(n)
    for k, off in enumerate((0, 8, 24)):
        a, b = at(off, n ** 3), at(off, n ** 3)
        a[:] = r.uniform(-1, 1, n ** 3) * 10.0 ** r.integers(-30, 30, n ** 3)
        a[:4] = np.inf, -np.inf, np.nan, -0.0
        b[:] = 7.0
        var = k % 2
        assert L.etd_set_field(g.ctx, var, a.ctypes.data_as(C.POINTER(C.c_double))) == 0
        assert L.etd_get_field(g.ctx, var, b.ctypes.data_as(C.POINTER(C.c_double))) == 0
        want = a if precision == 0 else a.astype(np.float32).astype(np.float64)
        assert np.array_equal(b.view(np.uint64), want.copy().view(np.uint64))
    g.close()


def test_boxes_round_trip():
    g = pyetd.Etd.from_dict(dict(small_params(n=66, nac=2), procs=(2, 1, 2)))
    r = np.random.default_rng(3)
    f = [r.uniform(-1, 1, (4, 66, 66, 66)) for _ in range(2)]
    for v in range(2):
        g.set_field(v, f[v])
    for v in range(2):
        assert np.array_equal(g.get_field(v), f[v])
    g.close()


def test_contexts_on_threads():
    """Contexts of several sizes read and set their fields from threads at once (they share pinned memory)."""
    import threading

    ns, bad = (100, 132, 68, 104, 128, 84), []

    def work(n):
        g = pyetd.Etd.from_dict(dict(small_params(n=n, nac=1), precision=2 if n % 8 else 0))
        for k in range(4):
            f = np.random.default_rng(n + k).integers(-1000, 1000, (n, n, n)).astype(float)
            g.set_field(0, f)
            if not np.array_equal(g.get_field(0), f):
                bad.append((n, k))
        g.close()

    th = [threading.Thread(target=work, args=(n,)) for n in ns]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
