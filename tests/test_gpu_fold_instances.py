"""GPU test of the folded products at one even and one odd edge of every
instance (rows in 1 to 17 tiles of 8), in both directions, against the dense
product, with the bound of test_gpu_fold.py."""
import numpy as np
import pytest

from test_gpu_fold import EPS, context, matrices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [n for rt in range(1, 18) for n in (16 * rt - 1, max(16 * rt, 34))])
def test_every_instance(n):
    g = context(n)
    u = np.random.default_rng(n).uniform(-1, 1, n ** 3)
    X = u.reshape(n * n, n).T
    for kind, A in matrices(n, 3).items():
        print(f"fold instance n={n} {kind}", flush=True)
        got = g.modeprod(A, u).reshape(n, n * n)
        bound = 2 * (n + 64) * EPS * (np.abs(A) @ np.abs(X)) + 64 * EPS * np.abs(A).max() * np.abs(X).sum(0)
        assert (np.abs(got - A @ X) <= bound).all()
    g.close()
