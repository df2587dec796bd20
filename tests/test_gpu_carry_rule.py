"""GPU test of when FP64 steps carry the AC spectrum: by size, unless
ETD_CARRY=1 (always) or 0 (never) says otherwise.  Small boxes that carry on
request equal the ones that transform u, to roundoff, and boxes on either side
of the line give the same fields whichever way they step."""
import os

import numpy as np
import pytest

import pyetd
from conftest import OMEGA_LANDAU, small_params

pytestmark = pytest.mark.gpu


def run(prm, env, steps, adaptive=False):
    if env is not None:
        os.environ["ETD_CARRY"] = env
    try:
        g = pyetd.Etd.from_dict(prm)
    finally:
        os.environ.pop("ETD_CARRY", None)
    for v in range(g.V):
        g.init_noise(v, 5 + v, 0.1 if v >= prm["nac"] else 0.0, 0.01)
    if adaptive:
        g.run_adaptive(t_end=1.0, dt0=0.005, dt_max=0.005, tol=1e9, energy_test=0, max_attempts=steps)
    else:
        g.step(steps)
    out = [g.get_field(v) for v in range(g.V)]
    ms, launches = g.time_steps(2, False)
    g.close()
    return out, launches[7] > 0  # class 7: the carried spectrum's correction


@pytest.mark.parametrize("adaptive", [False, True])
@pytest.mark.parametrize("case", [
    dict(n=16, nac=3, nch=1, etd2=0, elastic=1, aniso=0),
    dict(n=16, nac=2, nch=1, etd2=1, elastic=1, aniso=1),
    dict(n=20, nac=1, nch=0, etd2=0, elastic=0, aniso=2),
], ids=lambda c: "n{n}_ac{nac}_etd2{etd2}".format(**c))
def test_carried_on_request(case, adaptive):
    prm = small_params(dt=0.02, landau=OMEGA_LANDAU, KE=42.0, h=(1.0, 0.9, 1.1), **case)
    a, carried = run(prm, "1", 5, adaptive)
    b, never = run(prm, "0", 5, adaptive)
    assert carried and not never
    assert max(np.abs(x - y).max() for x, y in zip(a, b)) < 1e-12


@pytest.mark.parametrize("n,nac,etd2,periodic,carries", [
    (36, 4, 0, 1, False), (108, 4, 0, 1, False), (112, 4, 0, 1, True), (136, 1, 0, 1, False), (140, 1, 0, 1, True),
    (140, 4, 1, 1, False), (196, 4, 1, 1, True), (60, 4, 0, 0, False), (68, 4, 0, 0, True), (88, 4, 1, 0, False),
    (92, 4, 1, 0, True),
])
def test_the_line(n, nac, etd2, periodic, carries):
    prm = dict(small_params(n=n, nac=nac, etd2=etd2, dt=0.02, landau=(0.2, 3.0, 3.0)), periodic=periodic)
    a, carried = run(prm, None, 3)
    assert carried == carries
    b, _ = run(prm, "0" if carries else "1", 3)
    assert max(np.abs(x - y).max() for x, y in zip(a, b)) < 1e-12


def test_mixed_contexts_carry_at_any_size():
    assert run(dict(small_params(n=16, nac=2), precision=2), None, 2)[1]
