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

import oracle as O
import pyetd
from conftest import cubic_voigt, noise_fields, small_params

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


def voigt(kind):
    r = np.random.default_rng(4)
    if kind == "triclinic":
        A = r.uniform(-1, 1, (6, 6))
        return 40 * (A @ A.T / 6 + np.eye(6))
    return cubic_voigt(*{"isotropic": (134.0, 60.0, 37.0), "soft shear": (134.0, 110.0, 0.01)}.get(
        kind, (134.0, 110.0, 36.0)))


def exact_force(C2, eps0, fields):
    """felas on the interior in long double: DFT matrices and B_pq per point."""
    LD, N, nac = np.longdouble, fields[0].shape[0], len(fields)
    vg = np.array([[0, 5, 4], [5, 1, 3], [4, 3, 2]])
    C4 = C2[vg[:, :, None, None], vg[None, None]].astype(LD)
    eps = np.asarray(eps0).astype(LD)
    sig = np.einsum("ijkl,pkl->pij", C4, eps)
    t0 = np.einsum("pij,qij->pq", eps, sig)
    k = np.arange(N)
    k = np.where(k < N // 2, k, k - N).astype(LD)
    n = np.array(np.broadcast_arrays(k, k[:, None], k[:, None, None]))  # x, y, z
    n[1, 0, 0, 0] = 1
    n = n / np.sqrt((n ** 2).sum(0))
    G = np.einsum("ijkl,jabc,labc->ikabc", C4, n, n)
    cof = np.array([[G[(i + 1) % 3, (j + 1) % 3] * G[(i + 2) % 3, (j + 2) % 3]
                     - G[(i + 1) % 3, (j + 2) % 3] * G[(i + 2) % 3, (j + 1) % 3] for j in range(3)] for i in range(3)])
    om = cof.transpose(1, 0, 2, 3, 4) / sum(G[0, j] * cof[0, j] for j in range(3))
    turn = 2 * np.arctan2(LD(0), LD(-1)) * ((np.outer(np.arange(N), np.arange(N)) % N).astype(LD)) / N
    W = np.cos(turn) - 1j * np.sin(turn)

    def dft(x, w):
        return np.einsum("ai,bj,ck,ijk->abc", w, w, w, x, optimize=True)

    F = [dft(f.astype(np.clongdouble), W) for f in fields]
    b = np.einsum("qij,iabc->qjabc", sig, n)
    out = []
    for p in range(nac):
        c = np.einsum("jabc,jkabc->kabc", b[p], om)
        acc = sum((t0[p, q] - (c * b[q]).sum(0)) * F[q] for q in range(nac))
        out.append((dft(acc, W.conj()) / N ** 3).real)
    return out


@pytest.mark.parametrize("kind", ["isotropic", "triclinic", "soft shear", "cubic", "traceless"])
@pytest.mark.parametrize("nac", [7, 12])
def test_fp64_force_of_six_strains(nac, kind):
    """The FP64 force against a long double one: no further off than 1.5 times the oracle's FP64 transform per
    variant (the same roundings, two more for the six strains, other FFTs)."""
    prm = dict(small_params(n=20, nac=nac, elastic=1), C=voigt(kind))
    if kind == "traceless":
        prm["eps0"] = strains(kind, nac, np.random.default_rng(nac))
    o, g = O.Oracle(prm), pyetd.Etd.from_dict(prm)
    f = noise_fields(prm, amp=0.3)
    for v in range(nac):
        o.set_field(v, f[v])
        g.set_field(v, f[v])
    o.elastic()
    inner = (slice(2, -2),) * 3
    want = exact_force(prm["C"], prm["eps0"], [x[inner] for x in f])
    got = g.elastic()
    here = max(float(np.abs(got[p][inner] - want[p]).max()) for p in range(nac))
    oracle = max(float(np.abs(o.felas(p)[inner] - want[p]).max()) for p in range(nac))
    print(f"nac={nac} {kind}: {here:.2e}, oracle {oracle:.2e}", flush=True)
    assert here < 1.5 * oracle
    g.close()
