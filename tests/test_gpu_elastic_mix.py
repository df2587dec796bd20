"""GPU tests of elasticity with more than six variants, which transforms the
six strain components the variants span (etd_kernels.hip, launch_elastic),
against the oracle, which transforms every variant.

The smallest and largest numbers of variants that take this path (7, 16), an
odd one, edges with and without a two-stage FFT, several evaluations in a row
(ghost cells with two or three ghost coordinates hold variants of earlier
positions and, before variant 0, of the previous evaluation), physical sides,
a decomposed run, the steps that read the force in each place, the acceptance
energy, and an ensemble's replay.  Tolerances are those the same quantities
have with six variants or fewer."""
import numpy as np
import pytest

import oracle as O
import pyetd
from conftest import noise_fields, small_params

pytestmark = pytest.mark.gpu


def pair(prm, fields, precision=0):
    o, g = O.Oracle(prm), pyetd.Etd.from_dict(dict(prm, precision=precision))
    for v, f in enumerate(fields):
        o.set_field(v, f)
        g.set_field(v, f)
    return o, g


@pytest.mark.parametrize("precision,tol", [(0, 1e-12), (2, 1e-5)])
@pytest.mark.parametrize("nac,n", [(7, 12), (12, 20), (8, 36), (16, 24), (12, 52), (9, 40)])
def test_force_over_evaluations(nac, n, precision, tol):
    print(f"mixed elasticity nac={nac} n={n} precision={precision}", flush=True)
    prm = small_params(n=n, nac=nac, elastic=1, kk=(1.0, 1.0, 1.0))
    o, g = pair(prm, [f.astype(np.float32).astype(float) for f in noise_fields(prm, amp=0.4)], precision)
    for ev in range(3):
        o.transfer()
        g.transfer()
        o.elastic()
        got = g.elastic()
        scale = max(np.abs(o.felas(p)).max() for p in range(nac))
        for p in range(nac):
            assert np.abs(got[p] - o.felas(p)).max() < tol * scale, (ev, p)
        for v in range(nac):
            f = (o.get_field(v) * (1.1 + 0.05 * v) + 0.01).astype(np.float32).astype(float)
            o.set_field(v, f)
            g.set_field(v, f)
    g.close()


@pytest.mark.parametrize("precision,tol", [(0, 1e-10), (1, 1e-5), (2, 1e-5)])
@pytest.mark.parametrize("case", [
    dict(n=20, nac=7, nch=1, etd2=1, aniso=0),
    dict(n=36, nac=12, nch=1, etd2=0, aniso=0),
    dict(n=16, nac=8, nch=0, etd2=0, aniso=1),
    dict(n=20, nac=12, nch=0, etd2=1, aniso=2),
], ids=lambda c: "n{n}_ac{nac}_etd2{etd2}_an{aniso}".format(**c))
def test_steps(case, precision, tol):
    print(f"mixed elasticity steps {case} precision={precision}", flush=True)
    prm = small_params(elastic=1, dt=0.01, **case)
    o, g = pair(prm, noise_fields(prm, amp=0.1), precision)
    for _ in range(4):
        o.step()
        g.step()
    for v in range(prm["nac"] + prm["nch"]):
        assert np.abs(g.get_field(v) - o.get_field(v)).max() < tol
    g.close()


def test_physical_sides():
    prm = dict(small_params(n=20, nac=8, elastic=1), periodic=0)
    o = O.Oracle(prm)
    g = pyetd.Etd.from_dict(prm)
    for v, f in enumerate(noise_fields(prm, amp=0.3)):
        o.set_field(v, f)
        g.set_field(v, f)
    o.elastic()
    got = g.elastic()
    for p in range(8):
        ref = o.felas(p)
        assert np.abs(got[p] - ref).max() < 1e-12 * max(1e-3, np.abs(ref).max())
        assert (got[p][:2] == 0).all() and (got[p][:, -2:] == 0).all()
    o.step()
    g.step()
    assert max(np.abs(g.get_field(v) - o.get_field(v)).max() for v in range(8)) < 1e-10
    g.close()


def test_boxes():
    """2 x 2 x 2 boxes against the oracle's decomposed run."""
    prm = small_params(n=10, nac=7, elastic=1, dt=0.01, landau=(0.2, 3.0, 3.0), KE=3.2)
    G = O.OracleGroup(prm, (2, 2, 2))
    g = pyetd.Etd(pyetd.params_from_dict(dict(prm, procs=(2, 2, 2))))
    r = np.random.default_rng(8)
    for v in range(7):
        f = r.uniform(-0.2, 0.2, (8, 10, 10, 10))
        g.set_field(v, f)
        for b in range(8):
            G.box(b).set_field(v, f[b])
    for _ in range(3):
        G.step()
        g.step()
    for v in range(7):
        got = g.get_field(v)
        for b in range(8):
            assert np.abs(got[b] - G.box(b).get_field(v)).max() < 1e-10, (v, b)
    g.close()


def test_acceptance_energy():
    """The elastic part of both acceptance energies is ES/2 h^3 sum_p eta_p felas_p."""
    prm = small_params(n=16, nac=8, elastic=1, dt=0.01)
    f = noise_fields(prm, amp=0.2)
    for kind in (1, 0):
        E, u = [], None
        for el in (1, 0):
            _, g = pair(prm, f)
            st, log = g.run_adaptive(log_cap=4, t_end=0.01, dt0=0.01, tol=1e9, energy_test=0, energy_kind=kind,
                                     energy_elastic=el)
            assert st["accepted"] == 1
            E.append(log[0, 3])
            if el:
                u = [g.get_field(v) for v in range(8)]
            g.close()
        _, h = pair(prm, u)
        h.transfer()
        fel = h.elastic()
        inner = (slice(2, -2),) * 3
        e_el = 0.5 * sum(float((u[p][inner] * fel[p][inner]).sum()) for p in range(8))
        # the evaluation for the energy enters the ghost cells of the next
        # step's force; the run without it differs by that only
        assert abs(E[0] - E[1] - e_el) < 1e-3 * abs(e_el), (kind, E, e_el)
        h.close()


def test_ensemble_replay_equals_solo():
    prm = small_params(n=20, nac=8, elastic=1, dt=0.01)
    f = noise_fields(prm, amp=0.2)
    made = []
    for _ in range(2):
        g = pyetd.Etd.from_dict(prm, carry=False)
        for v, x in enumerate(f):
            g.set_field(v, x)
        g.step(1)
        made.append(g)
    with pytest.raises(pyetd.EtdError):  # the multiple of the ring's period it always asked for
        pyetd.Ensemble([made[0]], 4)
    E = pyetd.Ensemble([made[0]], 5)
    for _ in range(3):
        E.run(1)
        made[1].step(5)
        made[0].diag()
        for v in range(8):
            assert np.array_equal(made[0].get_field(v), made[1].get_field(v))
    E.close()
