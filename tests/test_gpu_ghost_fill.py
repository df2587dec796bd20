"""GPU test of the one-launch ghost fill against the oracle's sweeps, bit for
bit, with ghost cells that are no images beforehand: the smallest box it takes
(an interior of 2g cells: every row a source), one and two cells more, rows of
one to five passes of a wave, one and three ghost layers, several fields; and
of what it records for the carried spectrum (a carried step equals one that
transforms u only if every change is recorded)."""
import os

import numpy as np
import pytest

import oracle as O
import pyetd
from conftest import small_params

pytestmark = pytest.mark.gpu


EDGES = [(8, 2), (9, 2), (10, 2), (7, 2), (6, 1), (12, 3), (13, 3), (64, 2), (65, 2), (132, 2), (260, 2)]


@pytest.mark.parametrize("n,g,precision", [(n, g, p) for n, g in EDGES for p in ((0, 2) if n % 4 == 0 else (0,))])
def test_fill_equals_the_sweeps(n, g, precision):
    print(f"ghost fill n={n} g={g} precision={precision}", flush=True)
    c = pyetd.Etd.from_dict(dict(small_params(n=n, nac=3), g=g, precision=precision))
    r = np.random.default_rng(n)
    f = [r.uniform(-1, 1, (n, n, n)).astype(np.float32).astype(float) for _ in range(3)]
    for v in range(3):
        c.set_field(v, f[v])
    c.transfer()
    for v in range(3):
        assert np.array_equal(c.get_field(v), O.ghost_fill(f[v], g))
    c.close()


@pytest.mark.parametrize("n", [8, 9, 10, 21, 68])
def test_recorded_changes(n):
    prm = small_params(n=n, nac=2, dt=0.02)
    got = []
    for env in ("1", "0"):
        os.environ["ETD_CARRY"] = env
        try:
            c = pyetd.Etd.from_dict(prm)
        finally:
            os.environ.pop("ETD_CARRY", None)
        for v in range(2):
            c.set_field(v, np.random.default_rng(v).uniform(-0.3, 0.3, (n, n, n)))
        c.step(4)
        got.append([c.get_field(v) for v in range(2)])
        c.close()
    for a, b in zip(*got):
        assert np.abs(a - b).max() < 1e-12
