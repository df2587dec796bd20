"""GPU test of the FP64 transform's precision against a long double one, at
edges of every factor the two-stage kernels have (R1 = 16 and the others).

Tolerance: with every twiddle rounded once the rms error of a transform grows
as u sqrt(log2 of its points), u = 2^-53; a twiddle that is off by an ulp or
two, in a table or in a register DFT, repeats over the whole grid and takes
the error past that."""
import numpy as np
import pytest

import pyetd
from conftest import small_params

pytestmark = pytest.mark.gpu


def dft_matrix(N):
    LD = np.longdouble
    turn = 2 * np.arctan2(LD(0), LD(-1)) * ((np.outer(np.arange(N), np.arange(N)) % N).astype(LD)) / N
    return (np.cos(turn) - 1j * np.sin(turn)).astype(np.clongdouble)


@pytest.mark.parametrize("N", [16, 18, 20, 24, 27, 30, 36, 45, 50, 54, 60, 64, 72, 75, 81, 96])
def test_rms_error(N):
    g = pyetd.Etd.from_dict(small_params(n=N + 4, nac=1, elastic=1))
    r = np.random.default_rng(N)
    x = r.uniform(-1, 1, (N, N, N)) + 1j * r.uniform(-1, 1, (N, N, N))
    got = np.asarray(g.fft3d(x, 1)).reshape(N, N, N)
    g.close()
    W, ks = dft_matrix(N), [0, 1, N // 3, N // 2]
    want = np.stack([W @ p @ W.T for p in np.tensordot(W[ks], x.astype(np.clongdouble), (1, 0))])  # four planes
    err = float(np.sqrt((np.abs(got[ks] - want) ** 2).mean() / (np.abs(want) ** 2).mean()))
    bound = 2.0 ** -53 * np.sqrt(3 * np.log2(N))
    print(f"N={N}: {err:.2e}, bound {bound:.2e}", flush=True)
    assert err < bound
