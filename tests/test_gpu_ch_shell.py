"""GPU test of the CH nonlinear term on the cells near the box faces: edges at
which a wave holds cells of every kind, with and without inner points, on
periodic, decomposed and physical sides.

Tolerance: N is a second difference (12 / h^2 of t) of t = O(1), which itself
takes at most three outside values: some 60 terms of a few units with a few
roundings each, so 1e-12 of the larger of 1 and max |N| leaves more than a
factor of ten in FP64; FP32 storage rounds the result once (6e-8): 1e-6."""
import numpy as np
import pytest

import oracle as O
import pyetd
from conftest import small_params

pytestmark = pytest.mark.gpu


def fields(prm, P=1):
    rng = np.random.default_rng(prm["n"])
    n = prm["n"]
    return [rng.uniform(-0.3, 0.3, (P, n, n, n)).astype(np.float32).astype(np.float64)
            for _ in range(prm["nac"] + prm["nch"])]


@pytest.mark.parametrize("periodic", [1, 0])
@pytest.mark.parametrize("n,precision", [(9, 0), (12, 0), (13, 0), (21, 0), (66, 0), (12, 2), (20, 1), (68, 2)])
def test_one_box(n, periodic, precision):
    print(f"CH shell n={n} periodic={periodic} precision={precision}", flush=True)
    prm = dict(small_params(n=n, nac=1, nch=2, h=(0.9, 1.0, 1.2)), periodic=periodic, precision=precision)
    o = O.Oracle(dict(prm, precision=0))
    Vm, Vim, D = O.eigbasis(n, 3 if periodic else 0)
    g = pyetd.Etd(pyetd.params_from_dict(prm), Vm, Vim, D)
    for v, f in enumerate(fields(prm)):
        o.set_field(v, f[0])
        g.set_field(v, f[0])
    o.transfer()
    g.transfer()
    for v in (1, 2):
        ref = o.nonlinear(v)
        assert np.abs(g.nonlinear(v) - ref).max() < (1e-6 if precision else 1e-12) * max(1.0, np.abs(ref).max())
    g.close()


@pytest.mark.parametrize("procs,n", [((2, 1, 3), 9), ((1, 2, 2), 21)])
def test_boxes(procs, n):
    print(f"CH shell boxes {procs} n={n}", flush=True)
    prm = small_params(n=n, nac=1, nch=2, h=(0.9, 1.0, 1.2))
    P = int(np.prod(procs))
    G = O.OracleGroup(prm, procs)
    Vm, Vim, D = O.eigbasis(n, 3)
    g = pyetd.Etd(pyetd.params_from_dict(dict(prm, procs=procs)), Vm, Vim, D)
    for v, f in enumerate(fields(prm, P)):
        for b in range(P):
            G.box(b).set_field(v, f[b])
        g.set_field(v, f)
    G.transfer()
    g.transfer()
    for v in (1, 2):
        got = g.nonlinear(v)
        for b in range(P):
            ref = G.box(b).nonlinear(v)
            assert np.abs(got[b] - ref).max() < 1e-12 * max(1.0, np.abs(ref).max())
    g.close()
