"""GPU test of the mixed force's precision with more than six variants, which
are transformed as six strains (strain_basis): it is as near the FP64 force as
that of six variants, which are transformed one by one, whatever the strains
are.  Traceless strains are the hard ones: volume changes are the stiff
direction, so components that only cancel in the trace lose digits there.

Tolerance: a value passes some fourteen FP32 roundings on either way (three
axes there and back, packed and unpacked), two of them more with six strains;
sqrt(16 / 14) = 1.07, and the errors of two sets of variants spread by a tenth."""
import numpy as np
import pytest

import pyetd
from conftest import small_params

pytestmark = pytest.mark.gpu


def strains(kind, nac, rng):
    e = rng.uniform(-0.03, 0.03, (nac, 3, 3))
    e = 0.5 * (e + e.transpose(0, 2, 1))
    trace = np.trace(e, axis1=1, axis2=2)[:, None, None] * np.eye(3) / 3
    if kind == "traceless":
        e -= trace
    elif kind == "shear":
        e[:, range(3), range(3)] = 0
    elif kind == "volume":
        e = 0.02 * np.eye(3) + 0.05 * e
    return e


def error(prm, fields):
    force = []
    for precision in (0, 2):
        g = pyetd.Etd.from_dict(dict(prm, precision=precision))
        for v, f in enumerate(fields):
            g.set_field(v, f)
        force.append(np.array([f[2:-2, 2:-2, 2:-2] for f in g.elastic()]))
        g.close()
    return np.sqrt(((force[1] - force[0]) ** 2).mean() / (force[0] ** 2).mean())


@pytest.mark.parametrize("kind", ["any", "traceless", "shear", "volume"])
@pytest.mark.parametrize("n,nac", [(36, 12), (68, 12), (64, 16), (52, 7)])
def test_six_strains_are_as_accurate_as_six_variants(n, nac, kind):
    r = np.random.default_rng(n * 100 + nac)
    eps = strains(kind, nac, r)
    f = [r.uniform(-0.3, 0.3, (n, n, n)).astype(np.float32).astype(float) for _ in range(nac)]
    prm = small_params(n=n, nac=nac, elastic=1)
    many = error(dict(prm, eps0=eps), f)
    each = max(error(dict(small_params(n=n, nac=6, elastic=1), eps0=eps[k:k + 6]), f[k:k + 6]) for k in (0, nac - 6))
    print(f"n={n} nac={nac} {kind}: {many:.3e}, six variants {each:.3e}", flush=True)
    assert many < 1.2 * each
