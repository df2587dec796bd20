"""GPU test of the anisotropic gradient term's precision: N(u) of an AC field
in FP64 against a long double one, with equal and unequal spacing.

Tolerance: the oracle's error, which divides by 2h at every difference, and a
tenth: the term here has fewer roundings, and an rms over 36^3 values of both
is good to a percent."""
import numpy as np
import pytest

import oracle as O
import pyetd
from conftest import noise_fields, small_params

pytestmark = pytest.mark.gpu
LD = np.longdouble


def difference(f, axis, h):
    f = np.pad(f, 1)  # cells outside the box read 0
    lo, hi = [slice(1, -1)] * 3, [slice(1, -1)] * 3
    lo[axis], hi[axis] = slice(0, -2), slice(2, None)
    return (f[tuple(hi)] - f[tuple(lo)]) / (2 * h)


def exact(prm, fields, v):
    n = prm["n"]
    x = [f.astype(LD) for f in fields]
    u, s = x[v], sum(f * f for f in x)
    a2, a3, a4 = (LD(q) for q in prm["landau"])
    LE, e2, h = LD(prm["LE"]), LD(prm["epn2"]), [LD(q) for q in prm["h"]]
    out = LE * LD(prm["KE"]) * u - LE * (a2 * u - a3 * u * u + a4 * s * u)
    inside = (np.arange(n) - 2) % (n - 4) + 2  # periodic images
    for axis, hh in ((2, h[0]), (1, h[1]), (0, h[2])):
        for at, beyond in ((0, n - 5), (n - 1, 4)):  # the images of -1 and n
            ix = [inside] * 3
            ix[axis] = np.array([beyond])
            face = [slice(None)] * 3
            face[axis] = slice(at, at + 1)
            out[tuple(face)] += LE * e2 * u[np.ix_(*ix)] / hh ** 2
    g = [difference(u, 2, h[0]), -difference(u, 1, h[1]), -difference(u, 0, h[2])]
    L = prm["lam"][v].astype(LD)
    q = [sum(L[i, j] * g[j] for j in range(3)) for i in range(3)]
    return out - e2 * LE * (difference(q[0], 2, h[0]) - difference(q[1], 1, h[1]) - difference(q[2], 0, h[2]))


@pytest.mark.parametrize("kk", [1.0, 2.5])
@pytest.mark.parametrize("h", [(1.0, 1.0, 1.0), (1.0625,) * 3, (1.0, 0.9, 1.1), (1.3, 0.7, 1.25)])
def test_as_near_as_the_oracle(h, kk):
    prm = small_params(n=36, nac=3, aniso=1, h=h, kk=(kk,) * 3)
    o, g = O.Oracle(prm), pyetd.Etd.from_dict(prm)
    f = [O.ghost_fill(O.ghost_fill(O.ghost_fill(x, 2), 2), 2) for x in noise_fields(prm, amp=0.3)]  # all ghosts images
    for v in range(3):
        o.set_field(v, f[v])
        g.set_field(v, f[v])
    for v in range(3):
        want = exact(prm, f, v)
        err = [float(np.sqrt(((np.asarray(x).reshape(want.shape) - want) ** 2).mean() / (want ** 2).mean()))
               for x in (g.nonlinear(v), o.nonlinear(v))]
        print(f"h={h} kk={kk} field {v}: {err[0]:.3e}, oracle {err[1]:.3e}", flush=True)
        assert err[0] < 1.1 * err[1]
    g.close()
