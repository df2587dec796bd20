"""GPU test of the one-pass anisotropic gradient term: edges where a wave's
cells touch both ends of a row, more blocks than one box has, every field and
box in one launch, on periodic, decomposed and physical sides.

Tolerance: N is formed in FP64 from about 60 terms, the largest of size
max |Lambda| max |u| / h^2 (a few units); with the reciprocals of 2h each
contributes a few roundings of 2.2e-16, so 1e-13 of the larger of 1 and max
|N| leaves a factor of ten.  FP32 storage rounds N twice (before and after
the term): 1e-6 of the same leaves a factor of five."""
import numpy as np
import pytest

import oracle as O
import pyetd
from conftest import small_params

pytestmark = pytest.mark.gpu

LAM = np.array([[[1.3, 0.2, -0.1], [0.2, 0.8, 0.15], [-0.1, 0.15, 1.1]],
                [[0.7, -0.3, 0.25], [-0.3, 1.2, 0.05], [0.25, 0.05, 0.9]]])


def check(got, ref, precision):
    assert np.abs(got - ref).max() < (1e-6 if precision else 1e-13) * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("periodic", [1, 0])
@pytest.mark.parametrize("n,precision", [(10, 0), (13, 0), (20, 0), (68, 0), (12, 2), (20, 2), (36, 2)])
def test_one_box(n, periodic, precision):
    print(f"F2 n={n} periodic={periodic} precision={precision}", flush=True)
    prm = small_params(n=n, nac=2, aniso=1, h=(0.9, 1.0, 1.2))
    prm.update(lam=LAM, periodic=periodic, precision=precision)
    o = O.Oracle(dict(prm, precision=0))
    Vm, Vim, D = O.eigbasis(n, 3 if periodic else 0)
    g = pyetd.Etd(pyetd.params_from_dict(prm), Vm, Vim, D)
    rng = np.random.default_rng(n)
    for v in range(2):
        f = rng.uniform(-0.5, 0.5, (n, n, n)).astype(np.float32).astype(np.float64)
        o.set_field(v, f)
        g.set_field(v, f)
    o.transfer()
    g.transfer()
    for v in range(2):
        check(g.nonlinear(v), o.nonlinear(v), precision)
    g.close()


@pytest.mark.parametrize("procs,n", [((2, 1, 3), 13), ((1, 2, 1), 36)])
def test_boxes(procs, n):
    print(f"F2 boxes {procs} n={n}", flush=True)
    prm = small_params(n=n, nac=2, nch=1, aniso=1, h=(0.9, 1.0, 1.2))
    prm.update(lam=LAM)
    P = int(np.prod(procs))
    G = O.OracleGroup(prm, procs)
    Vm, Vim, D = O.eigbasis(n, 3)
    g = pyetd.Etd(pyetd.params_from_dict(dict(prm, procs=procs)), Vm, Vim, D)
    rng = np.random.default_rng(n)
    for v in range(3):
        f = rng.uniform(-0.5, 0.5, (P, n, n, n))
        for b in range(P):
            G.box(b).set_field(v, f[b])
        g.set_field(v, f)
    G.transfer()
    g.transfer()
    for v in range(2):
        got = g.nonlinear(v)
        for b in range(P):
            check(got[b], G.box(b).nonlinear(v), 0)
    g.close()
