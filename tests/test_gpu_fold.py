"""GPU test of the folded FP64 mode products (a basis whose modes alternate in
parity) against a dense product in extended precision and the full-size
kernel, through the C ABI.

Edges: the smallest that fold (odd 9, even 34) and the ones below, one and two
K steps past a chunk of 16 pairs, every remainder of the row tiles, odd edges (8-byte loads,
a middle row), the largest edge; columns that do not fill the last workgroup.
Tolerance: an n-term dot product in FP64 is within n eps sum |a||x| of the
exact one, the fold adds one rounding and the symmetrised matrix 64 eps."""
import numpy as np
import pytest

import pyetd
from conftest import small_params

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def context(n):
    return pyetd.Etd.from_dict(small_params(n=n, nac=1))


def variant(g, v):
    t = g.get_tuning()
    t.mp_variant = v
    g.set_tuning(t)


def matrices(n, bcid):
    V, Vi, _ = pyetd.eigbasis(n, bcid)
    r = np.random.default_rng(n)
    # parity along the columns (forward), along the rows only (backward)
    return {"forward": Vi * r.uniform(0.5, 2, n)[:, None], "backward": V * r.uniform(0.5, 2, n)[None, :],
            "none": r.uniform(-1, 1, (n, n))}


@pytest.mark.parametrize("bcid", [3, 0])
@pytest.mark.parametrize("n", [7, 8, 9, 11, 15, 17, 31, 32, 33, 34, 36, 41, 49, 66, 68, 97, 104, 132])
def test_folded_products(n, bcid):
    g = context(n)
    u = np.random.default_rng(5).uniform(-1, 1, n ** 3)
    X = u.reshape(n * n, n).T  # [k][column]
    for kind, A in matrices(n, bcid).items():
        print(f"fold n={n} id={bcid} {kind}", flush=True)
        ref = (A.astype(np.longdouble) @ X.astype(np.longdouble)).astype(float)
        bound = (n + 64) * EPS * (np.abs(A) @ np.abs(X)) + 64 * EPS * np.abs(A).max() * np.abs(X).sum(0)
        variant(g, 1)
        got = g.modeprod(A, u).reshape(n, n * n)  # rotated: out[column + n^2 m]
        assert (np.abs(got - ref) <= bound).all()
        variant(g, 4)
        full = g.modeprod(A, u).reshape(n, n * n)
        assert (np.abs(got - full) <= 2 * bound).all()
        if n % 2 and (kind == "none" or n < 8):
            assert np.array_equal(got, full)  # the full-size kernel (odd edges have one tiling of it)
    g.close()


@pytest.mark.parametrize("n", [196, 260, 271, 272])
def test_folded_products_largest(n):
    g = context(n)
    u = np.random.default_rng(6).uniform(-1, 1, n ** 3)
    X = u.reshape(n * n, n).T
    for kind, A in matrices(n, 3).items():
        print(f"fold n={n} {kind}", flush=True)
        ref = A @ X
        got = g.modeprod(A, u).reshape(n, n * n)
        bound = 2 * (n + 64) * EPS * (np.abs(A) @ np.abs(X)) + 64 * EPS * np.abs(A).max() * np.abs(X).sum(0)
        assert (np.abs(got - ref) <= bound).all()
    g.close()


@pytest.mark.parametrize("n,periodic,etd2,nac,nch", [(34, 1, 1, 2, 1), (21, 1, 1, 2, 1), (36, 0, 1, 1, 1), (23, 0, 0, 3, 0)])
def test_folded_steps_equal_full_products(n, periodic, etd2, nac, nch):
    """Whole steps (several fields a launch, the accumulating backward product of the ETD2 corrector)."""
    prm = dict(small_params(n=n, nac=nac, nch=nch, etd2=etd2), periodic=periodic)
    got = []
    for v in (1, 4):
        g = pyetd.Etd.from_dict(prm)
        variant(g, v)
        for k in range(g.V):
            g.init_noise(k, 11 + k, 0.1, 0.2)
        print(f"fold steps n={n} periodic={periodic} variant={v}", flush=True)
        g.step(4)
        got.append([g.get_field(k) for k in range(g.V)])
        g.close()
    for a, b in zip(*got):
        assert np.abs(a - b).max() < 1e-12
