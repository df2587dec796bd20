"""GPU tests of the carried spectrum at the small sizes the oracle can follow,
where FP64 contexts would not carry by themselves (carry_pays): the checks of
test_gpu_carry.py and test_gpu_adaptive.py with ETD_CARRY=1 on the carried
side, which is seen to carry."""
import os

import pytest

import oracle as O
import pyetd
import test_gpu_adaptive as A
import test_gpu_carry as T

pytestmark = pytest.mark.gpu


def make(prm, carry):
    os.environ["ETD_CARRY"] = "1" if carry else "0"
    try:
        Vm, Vim, D = O.eigbasis(prm["n"], 3 if prm.get("periodic", 1) else 0)
        return pyetd.Etd(pyetd.params_from_dict(prm), Vm, Vim, D)
    finally:
        os.environ.pop("ETD_CARRY", None)


@pytest.fixture(autouse=True)
def forced(monkeypatch):
    seen = []

    def gpu(prm, carry):
        probe = make(prm, carry)
        launches = probe.time_steps(2, False)[1]
        probe.close()
        assert (launches[7] > 0) == carry  # class 7: the carried spectrum's correction
        seen.append(carry)
        return make(prm, carry)

    def gpu_fields(prm, fields, carry=True):
        g = gpu(prm, carry)
        for v, f in enumerate(fields):
            g.set_field(v, f)
        return g

    monkeypatch.setattr(T, "gpu", gpu)
    monkeypatch.setattr(A, "gpu", gpu_fields)
    yield
    assert True in seen


@pytest.mark.parametrize("case", [c for c in T.CASES if c["precision"] == 0],
                         ids=lambda c: "n{n}_ac{nac}_etd2{etd2}_el{elastic}_an{aniso}".format(**c))
def test_steps(case):
    T.test_carried_steps_match_transformed_steps_and_oracle(case)


def test_long_run():
    T.test_carried_steps_do_not_drift_over_a_long_run()


def test_set_field():
    T.test_setting_a_field_drops_the_carried_spectrum()


@pytest.mark.parametrize("extrapolate,etd2", [(1, 0), (0, 0), (1, 1)])
def test_adaptive(extrapolate, etd2):
    A.test_carried_attempts_match_transformed_attempts(0, extrapolate, etd2)
