"""GPU tests of the two-stage line FFT on every edge it is built for besides
16 R2, against numpy, and of the elastic force through it (the pack and unpack
are part of its first and last pass) against the oracle: last groups of lines
that are short (odd edges, 18, 30, ...), more threads than stage-one lanes
(R1 > R2), one to six transformed fields and the six-component pack.

FP64 within 1e-12 of the largest value (numpy's own transform is as far from
exact), FP32 within 2e-6, as the other edges."""
import numpy as np
import pytest

import oracle as O
import pyetd
from conftest import noise_fields, small_params

pytestmark = pytest.mark.gpu

EDGES = [18, 20, 24, 25, 27, 30, 36, 40, 45, 50, 54, 60, 72, 75, 81, 90, 100, 108, 120, 135, 150, 180]


@pytest.mark.parametrize("N,precision", [(N, p) for N in EDGES for p in ((0, 2) if N % 4 == 0 else (0,))])
def test_fft3d(N, precision):
    print(f"fft2 N={N} precision={precision}", flush=True)
    g = pyetd.Etd.from_dict(dict(small_params(n=N + 4, nac=1, elastic=1), precision=precision))
    r = np.random.default_rng(N)
    x = (r.standard_normal((N, N, N)) + 1j * r.standard_normal((N, N, N))).astype(np.complex64).astype(complex)
    ref = np.fft.fftn(x)
    tol = 1e-12 if precision == 0 else 2e-6
    assert np.abs(g.fft3d(x, 1) - ref).max() < tol * np.abs(ref).max()
    assert np.abs(g.fft3d(ref, -1) / N ** 3 - x).max() < tol * np.abs(x).max()
    g.close()


@pytest.mark.parametrize("N,nac,precision", [
    (18, 1, 0), (20, 2, 0), (20, 5, 2), (24, 4, 1), (25, 3, 0), (27, 4, 0), (30, 6, 0), (36, 4, 2), (40, 3, 2),
    (45, 4, 0), (50, 1, 0), (54, 4, 0), (60, 4, 2), (72, 2, 0),
    (18, 7, 0), (25, 8, 0), (36, 12, 2), (45, 7, 0), (60, 12, 1),
])
def test_force(N, nac, precision):
    print(f"fft2 force N={N} nac={nac} precision={precision}", flush=True)
    prm = small_params(n=N + 4, nac=nac, elastic=1)
    o, g = O.Oracle(prm), pyetd.Etd.from_dict(dict(prm, precision=precision))
    for v, f in enumerate(noise_fields(prm, amp=0.4)):
        f = f.astype(np.float32).astype(float)
        o.set_field(v, f)
        g.set_field(v, f)
    for ev in range(2):
        o.transfer()
        g.transfer()
        o.elastic()
        got = g.elastic()
        scale = max(np.abs(o.felas(p)).max() for p in range(nac))
        for p in range(nac):
            assert np.abs(got[p] - o.felas(p)).max() < (1e-12 if precision == 0 else 1e-5) * scale, (ev, p)
    g.close()


@pytest.mark.parametrize("N", [36, 45])
def test_boxes(N):
    """A decomposed run's global grid (2N = 72, 90) through its separate pack and unpack."""
    prm = small_params(n=N + 4, nac=2, elastic=1)
    G = O.OracleGroup(prm, (2, 2, 2))
    g = pyetd.Etd(pyetd.params_from_dict(dict(prm, procs=(2, 2, 2))))
    r = np.random.default_rng(2)
    for v in range(2):
        f = r.uniform(-0.3, 0.3, (8,) + (N + 4,) * 3)
        g.set_field(v, f)
        for b in range(8):
            G.box(b).set_field(v, f[b])
    G.transfer()
    g.transfer()
    G.elastic()
    got = g.elastic()
    for p in range(2):
        for b in range(8):
            ref = G.box(b).felas(p)
            assert np.abs(got[p, b] - ref).max() < 1e-12 * np.abs(ref).max()
    g.close()
