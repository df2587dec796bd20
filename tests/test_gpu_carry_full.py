"""GPU test of when FP64 steps carry the AC spectrum where the mode products
are full-size: a basis without parity to rounding, as one read from files, or
another product variant chosen, also between steps.  Transforming u costs more
there, so smaller boxes carry than with folded products."""
import numpy as np
import pytest

import pyetd
from conftest import small_params

pytestmark = pytest.mark.gpu


def context(prm, noisy):
    V, Vi, D = pyetd.eigbasis(prm["n"], 3 if prm["periodic"] else 0)
    if noisy:  # files carry about 1e-12
        r = np.random.default_rng(3)
        V, Vi = (A + 1e-12 * r.uniform(-1, 1, A.shape) for A in (V, Vi))
    g = pyetd.Etd(pyetd.params_from_dict(prm), V, Vi, D)
    for v in range(g.V):
        g.init_noise(v, 5 + v, 0.0, 0.01)
    return g


def carries(g):
    return g.time_steps(2, False)[1][7] > 0  # class 7: the carried spectrum's correction


def variant(g, v):
    t = g.get_tuning()
    t.mp_variant = v
    g.set_tuning(t)


@pytest.mark.parametrize("noisy", [True, False])
@pytest.mark.parametrize("n,nac,etd2,periodic,full", [
    (84, 4, 0, 1, False), (92, 4, 0, 1, True), (132, 1, 0, 1, True), (79, 4, 0, 1, False), (81, 4, 0, 1, True),
    (128, 4, 1, 1, False), (132, 4, 1, 1, True), (60, 4, 0, 0, False), (64, 4, 0, 0, True), (72, 4, 1, 0, False),
    (76, 4, 1, 0, True),
])
def test_the_line(n, nac, etd2, periodic, full, noisy):
    print(f"carry by full products n={n} nac={nac} etd2={etd2} periodic={periodic} noisy={noisy}", flush=True)
    prm = dict(small_params(n=n, nac=nac, etd2=etd2, dt=0.02, landau=(0.2, 3.0, 3.0)), periodic=periodic)
    g = context(prm, noisy)
    if not noisy:
        variant(g, 4)
    assert carries(g) == full
    g.close()


def test_variant_changed_between_steps():
    """Folded products do not carry at this size, full ones do: the steps before and after a change are the same
    as without one, to rounding."""
    prm = dict(small_params(n=92, nac=4, dt=0.02, landau=(0.2, 3.0, 3.0)), periodic=1)
    a, b = context(prm, False), context(prm, False)
    for v in (1, 4, 1, 4, 4, 1):
        variant(a, v)
        a.step(2)
        b.step(2)
    for k in range(4):
        assert np.abs(a.get_field(k) - b.get_field(k)).max() < 1e-12
    variant(a, 4)
    assert carries(a) and not carries(b)
    a.close()
    b.close()
