"""Methods that a program replaced, on the class or on one simulator, before or
after the simulator was made, are called by step() and simulate() as often as the
loop over the substeps calls them."""

import functools

import numpy as np
import pytest

from tests._cases import state
from tests.test_gpu_step import BOUNDARIES, make

pytestmark = pytest.mark.gpu

DT = np.float32(2.0 ** -5)

SCHEMES = [("kp07_dimsplit", "fast"), ("ee2d_kp07_dimsplit", "exact"), ("kp07", "fast")]


def new(ctx, scheme, math):
    return make(ctx, scheme, state(scheme, 40, 30, seed=1), 40, 30, BOUNDARIES["periodic"], math)


def counted(function, calls):
    @functools.wraps(function)
    def call(*args, **kw):
        calls.append(0)
        return function(*args, **kw)
    return call


# calls of a step: two substeps, each with the arguments of two states
CALLS = {"substep": 2, "substepDimsplit": 2, "_launch": 2, "_field_args": 4, "cfl_pointer": 2}


@pytest.mark.parametrize("scheme,math,name", [(s, m, n) for s, m in SCHEMES for n in sorted(CALLS)
                                              if (s, n) != ("kp07", "substepDimsplit")])
def test_replaced_on_the_class_or_the_simulator(ctx, scheme, math, name, monkeypatch):
    a, b, plain = (new(ctx, scheme, math) for _ in range(3))
    print("case replaced", scheme, math, name, flush=True)
    calls = []
    setattr(a, name, counted(getattr(a, name), calls))
    a.step(DT)
    assert len(calls) == CALLS[name]
    a.simulate(float(3 * DT), DT)
    assert len(calls) == 4 * CALLS[name]
    calls.clear()
    monkeypatch.setattr(type(b), name, counted(getattr(type(b), name), calls))
    b.step(DT)
    assert len(calls) == CALLS[name]
    b.simulate(float(2 * DT), DT)
    assert len(calls) == 3 * CALLS[name]
    monkeypatch.undo()
    b.step(DT)
    for _ in range(4):
        plain.step(DT)
    for x, y, z in zip(a.download(), b.download(), plain.download()):
        assert np.array_equal(x, z) and np.array_equal(y, z)


@pytest.mark.parametrize("where", ["class", "simulator"])
@pytest.mark.parametrize("name,calls_a_step", [("substep", 2), ("full_exchange", 2), ("sim._launch", 2)])
def test_replaced_in_an_mpi_simulator(ctx, name, calls_a_step, where, monkeypatch):
    from finitevolumegpu_amd.MPISimulator import MPISimulator
    a, plain = (MPISimulator(new(ctx, "ee2d_kp07_dimsplit", "fast")) for _ in range(2))
    owner = a.sim if name.startswith("sim.") else a
    name = name.split(".")[-1]
    owner = type(owner) if where == "class" else owner
    calls = []
    monkeypatch.setattr(owner, name, counted(getattr(owner, name), calls))
    print("case replaced mpi", name, where, flush=True)
    for _ in range(3):
        a.step(DT)
    assert len(calls) == 3 * calls_a_step
    monkeypatch.undo()
    for _ in range(3):
        plain.step(DT)
    assert all(np.array_equal(x, y) for x, y in zip(a.download(), plain.download()))
