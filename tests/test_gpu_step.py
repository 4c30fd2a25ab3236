"""Simulator.step (one library call, one launch for the slope schemes and the
two-stage KP07 in fast arithmetic) against its two substeps run one by one: the fields and the CFL
minimum are equal bitwise.  Sizes at the edges of a strip of the whole-step
march (56 output columns, 120 with two columns per lane), smallest sides,
segments as short as they may be, and every kind of edge."""

import itertools

import numpy as np
import pytest

from oracle import fv_oracle as O
from tests._cases import make_gpu_sim, state

pytestmark = pytest.mark.gpu

R, P, F, D = O.REFLECTIVE, O.PERIODIC, O.OUTFLOW, O.DIRICHLET

BOUNDARIES = {
    "reflective": O.pack_bc(R, R, R, R),
    "periodic": O.pack_bc(P, P, P, P),
    "outflow": O.pack_bc(F, F, F, F),
    "mixed": O.pack_bc(R, F, F, R),
    "channel": O.pack_bc(F, R, P, P),
}

SIZES = [(8, 8), (9, 11), (55, 12), (56, 8), (57, 30), (59, 9), (60, 64), (113, 65), (120, 17), (121, 40), (123, 8),
         (241, 133)]

CASES = [("kp07_dimsplit", "fast"), ("hll2", "fast"), ("ee2d_kp07_dimsplit", "fast"), ("kp07", "fast"),
         ("ee2d_kp07_dimsplit", "exact"), ("waf", "exact"), ("kp07", "exact")]


def make(ctx, scheme, fields, nx, ny, bc, math="fast", **kw):
    if scheme != "kp07":  # the unsplit scheme, two Runge-Kutta stages
        return make_gpu_sim(ctx, scheme, fields, nx, ny, 1.0, 1.0, bc, math=math, **kw)
    from finitevolumegpu_amd.KP07 import KP07
    from finitevolumegpu_amd.Simulator import BoundaryCondition
    return KP07(ctx, *fields, nx, ny, 1.0, 1.0, 9.81, boundary_conditions=BoundaryCondition(
        BoundaryCondition.getTypes(bc)), math=math, **kw)


def run_pair(ctx, scheme, nx, ny, bc, math, steps=3, **kw):
    fields = state(scheme, nx, ny, seed=nx + 7 * ny)
    a = make(ctx, scheme, fields, nx, ny, bc, math, **kw)
    b = make(ctx, scheme, fields, nx, ny, bc, math, **kw)
    dt = np.float32(0.05) if scheme == "ee2d_kp07_dimsplit" else np.float32(0.9 * a.computeDt())
    for n in range(steps):
        a.step(dt)
        for i in range(2):
            b.substep(dt, i)
        assert a.computeDt() == b.computeDt(), (n, a.computeDt(), b.computeDt())
        for k, (x, y) in enumerate(zip(a.download(), b.download())):
            assert np.array_equal(x, y), (n, k, np.argwhere(x != y)[:5].tolist())
    return a, b, dt


@pytest.mark.parametrize("bc", sorted(BOUNDARIES))
@pytest.mark.parametrize("scheme,math", CASES)
def test_step_equals_its_substeps(ctx, scheme, math, bc):
    sizes = SIZES if math == "fast" else SIZES[-2:]
    for nx, ny in sizes:
        print("case step", scheme, math, bc, nx, ny, flush=True)
        run_pair(ctx, scheme, nx, ny, BOUNDARIES[bc], math)


@pytest.mark.parametrize("scheme", ["kp07_dimsplit", "ee2d_kp07_dimsplit", "kp07"])
def test_step_with_every_combination_of_edges(ctx, scheme):
    """All 256 combinations of the four edge kinds, those that take one launch
    and those that take two."""
    nx, ny = 61, 18
    frame = (1.05, 0.01, -0.01, 6.5)
    fields = state(scheme, nx, ny, seed=4)
    pads = []
    for k, f in enumerate(fields):
        pad = np.full((ny + 4, nx + 4), frame[k], dtype=np.float32)
        pad[2:-2, 2:-2] = f
        pads.append(pad)
    print("case step edges", scheme, flush=True)
    for code in itertools.product((D, P, R, F), repeat=4):
        out = []
        for whole in (True, False):
            sim = make(ctx, scheme, fields, nx, ny, O.pack_bc(*code))
            for buf in (sim.u0, sim.u1):  # ghost memory that Dirichlet edges read
                for k, pad in enumerate(pads):
                    buf[k].upload(sim.stream, pad, extent=[0, 0, nx + 4, ny + 4])
            if whole:
                sim.step(np.float32(0.04))
            else:
                sim.substep(np.float32(0.04), 0)
                sim.substep(np.float32(0.04), 1)
            out.append(sim.download() + [np.float32(sim.computeDt())])
        assert all(np.array_equal(x, y) for x, y in zip(*out)), code


@pytest.mark.parametrize("scheme", ["kp07_dimsplit", "ee2d_kp07_dimsplit", "kp07"])
@pytest.mark.parametrize("tile_rows,waves", [(4, 4), (5, 1), (9, 2), (3, 4), (64, 3)])
def test_step_of_any_launch_shape(ctx, scheme, tile_rows, waves):
    for nx, ny in ((70, 45), (250, 61)):
        print("case step shape", scheme, nx, ny, tile_rows, waves, flush=True)
        run_pair(ctx, scheme, nx, ny, BOUNDARIES["mixed"], "fast", tile_rows=tile_rows, waves_per_block=waves)


@pytest.mark.parametrize("scheme,nx,ny", [("kp07_dimsplit", 4096, 2050), ("hll2", 2300, 4095),
                                          ("ee2d_kp07_dimsplit", 3001, 4032), ("kp07", 3000, 4000)])
@pytest.mark.parametrize("bc", ["mixed", "periodic"])
def test_step_with_the_round_weighted_split(ctx, scheme, nx, ny, bc):
    print("case step rounds", scheme, nx, ny, bc, flush=True)
    run_pair(ctx, scheme, nx, ny, BOUNDARIES[bc], "fast", steps=2)


def test_step_and_substeps_in_turn(ctx):
    """Whole steps and single substeps of one simulator, in any order, leave
    the CFL minimum of the last step and the same state."""
    a, b, dt = run_pair(ctx, "kp07_dimsplit", 64, 40, BOUNDARIES["reflective"], "fast")
    for whole in (False, True, True, False, True):
        if whole:
            a.step(dt)
        else:
            a.substep(dt, 0)
            a.substep(dt, 1)
        b.substep(dt, 0)
        b.substep(dt, 1)
        assert a.computeDt() == b.computeDt()
    assert all(np.array_equal(x, y) for x, y in zip(a.download(), b.download()))


def test_dirichlet_edges_read_both_buffers(ctx):
    """A Dirichlet edge reads each substep's own input buffer, so its step
    takes the substep launches: different ghost values in the two buffers."""
    nx, ny = 70, 50
    bc = O.pack_bc(D, R, R, D)
    sims = [make_gpu_sim(ctx, "kp07_dimsplit", state("kp07_dimsplit", nx, ny, 5), nx, ny, 1.0, 1.0, bc)
            for _ in range(2)]
    for sim in sims:
        for j, buf in enumerate((sim.u0, sim.u1)):
            for k, v in enumerate((1.0 + 0.1 * j, 0.02 * j, -0.01)):
                pad = np.full((ny + 4, nx + 4), v, dtype=np.float32)
                pad[2:-2, 2:-2] = buf[k].download(sim.stream)
                buf[k].upload(sim.stream, pad, extent=[0, 0, nx + 4, ny + 4])
    for _ in range(4):
        sims[0].step(np.float32(0.08))
        for i in range(2):
            sims[1].substep(np.float32(0.08), i)
    assert all(np.array_equal(x, y) for x, y in zip(sims[0].download(), sims[1].download()))
    assert sims[0].computeDt() == sims[1].computeDt()


def test_subclass_with_its_own_substep_is_called(ctx):
    from finitevolumegpu_amd.KP07_dimsplit import KP07_dimsplit

    class Counting(KP07_dimsplit):
        calls = 0

        def substep(self, dt, step_number):
            self.calls += 1
            super().substep(dt, step_number)

    sim = Counting(ctx, *state("kp07_dimsplit", 32, 32, 1), 32, 32, 1.0, 1.0, 9.81)
    sim.step(np.float32(0.05))
    assert sim.calls == 2


@pytest.mark.parametrize("math", ["fast", "exact"])
def test_mpi_step_equals_exchange_between_substeps(ctx, math):
    from finitevolumegpu_amd.MPISimulator import MPISimulator
    nx, ny = 130, 75
    sims = [MPISimulator(make_gpu_sim(ctx, "ee2d_kp07_dimsplit", state("ee2d_kp07_dimsplit", nx, ny, 2), nx, ny, 1.0,
                                      1.0, BOUNDARIES["channel"], math=math)) for _ in range(2)]
    dt = np.float32(0.05)
    for _ in range(3):
        sims[0].step(dt)
        for i in range(2):
            sims[1].substep(dt, i)
        padded = [[v.download(s.stream, extent=[0, 0, nx + 4, ny + 4]) for v in s.getOutput().gpu_variables]
                  for s in sims]
        assert all(np.array_equal(x, y) for x, y in zip(*padded))
    assert sims[0].computeDt() == sims[1].computeDt()
    assert sims[0].profiling_data_mpi["n_time_steps"] == sims[1].profiling_data_mpi["n_time_steps"]


@pytest.mark.parametrize("scheme", ["LxF", "HLL", "FORCE"])
@pytest.mark.parametrize("bc", sorted(BOUNDARIES) + ["one-sided"])
def test_first_order_with_two_columns_per_lane(ctx, scheme, bc):
    """One-row segments make enough waves for two columns per lane, 64-row
    segments leave one: the same fields, at the edges of 124-column strips."""
    import importlib
    from finitevolumegpu_amd.Simulator import BoundaryCondition
    cls = getattr(importlib.import_module("finitevolumegpu_amd." + scheme), scheme)
    code = O.pack_bc(P, R, R, P) if bc == "one-sided" else BOUNDARIES[bc]
    edges = BoundaryCondition(BoundaryCondition.getTypes(code))
    ny = 1100
    for nx in (2, 61, 122, 123, 124, 125, 247, 248):
        print("case two columns", scheme, bc, nx, flush=True)
        fields = state("kp07_dimsplit", nx, ny, seed=nx)
        sims = [cls(ctx, *fields, nx, ny, 1.0, 1.0, 9.81, boundary_conditions=edges, tile_rows=rows)
                for rows in (1, 64)]
        dt = np.float32(0.5 * sims[0].computeDt())
        for _ in range(2):
            for sim in sims:
                sim.step(dt)
        assert all(np.array_equal(x, y) for x, y in zip(*[s.download() for s in sims])), nx
        assert sims[0].computeDt() == sims[1].computeDt()


def _ensemble_specs(codes, sizes, seed):
    specs = []
    for j, ((nx, ny), code) in enumerate(zip(sizes, codes)):
        specs.append({"fields": state("kp07_dimsplit", nx, ny, seed + j), "nx": nx, "ny": ny, "dx": 1.0, "dy": 1.0,
                      "g": 9.81, "t_end": 1.3 + 0.4 * j, "bc": code})
    return specs


@pytest.mark.parametrize("scheme", ["kp07_dimsplit", "hll2"])
@pytest.mark.parametrize("steps_per_graph,seg_rows", [(3, None), (4, 5)])
def test_ensemble_of_whole_steps_equals_plain_runs(ctx, scheme, steps_per_graph, seg_rows):
    """Instances that finish after odd and even step counts, in blocks of odd
    and even length: each equals its plain run, also its non-finite count's
    buffer.  An instance with a Dirichlet edge joining midway turns the whole
    ensemble to substeps, with every instance's state where it was."""
    from finitevolumegpu_amd.Ensemble import Ensemble
    sizes = [(8, 8), (57, 33), (113, 65), (70, 120)]
    codes = [BOUNDARIES[k] for k in ("reflective", "mixed", "periodic", "outflow")]
    specs = _ensemble_specs(codes, sizes, 11)
    late = _ensemble_specs([O.pack_bc(R, R, P, R)], [(40, 30)], 50)[0]  # one-sided periodic: substeps
    late["t_end"] = 1.0
    ens = Ensemble(ctx, scheme, specs, steps_per_graph=steps_per_graph, seg_rows=seg_rows, capacity=6)
    ens.advance()
    assert ens.whole_steps
    slot = ens.add(late)
    ens.advance()
    assert not ens.whole_steps
    ens.remove(slot) if slot in ens.finished() else None
    ens.run()
    for i, spec in list(enumerate(specs)) + [(slot, late)]:
        if not ens.live[i]:
            continue
        sim = make(ctx, scheme, spec["fields"], spec["nx"], spec["ny"], spec["bc"])
        sim.simulate(spec["t_end"])
        t, nt = ens.state(i)
        assert nt == sim.simSteps() and t == sim.simTime()
        assert all(np.array_equal(x, y) for x, y in zip(ens.download(i), sim.download())), i
    assert (ens.nonfinite_counts(range(len(specs))) == 0).all()
    ens.close()
    # and with whole steps to the end
    ens = Ensemble(ctx, scheme, specs, steps_per_graph=steps_per_graph, seg_rows=seg_rows)
    ens.run()
    assert ens.whole_steps
    parities = set()
    for i, spec in enumerate(specs):
        sim = make(ctx, scheme, spec["fields"], spec["nx"], spec["ny"], spec["bc"])
        sim.simulate(spec["t_end"])
        parities.add(sim.simSteps() % 2)
        assert ens.state(i)[1] == sim.simSteps()
        assert all(np.array_equal(x, y) for x, y in zip(ens.download(i), sim.download())), i
    assert parities == {0, 1}
    ens.close()


RUNS = [("kp07_dimsplit", "fast"), ("hll2", "fast"), ("waf", "exact"), ("ee2d_kp07_dimsplit", "exact"),
        ("kp07", "fast")]


def step_loop(sim, t, dt=None):
    """The loop of simulate(), a step at a time."""
    t_end = sim.simTime() + t
    sim.dt = sim.dt if dt is None else dt
    while sim.simTime() < t_end:
        if dt is None and sim.simSteps() % 100 == 0:
            sim.dt = sim.computeDt() * sim.cfl_scale
        sim.step(np.float32(min(sim.dt, t_end - sim.simTime())))


@pytest.mark.parametrize("given", [None, float, np.float32])
@pytest.mark.parametrize("scheme,math", RUNS)
def test_simulate_equals_the_loop_of_steps(ctx, scheme, math, given):
    """Runs of steps in one library call: across refreshes of dt, ending inside
    one, on one (odd numbers of steps) and not at all, and with substeps between."""
    nx, ny = 61, 34
    fields = state(scheme, nx, ny, seed=8)
    a, b = (make(ctx, scheme, fields, nx, ny, BOUNDARIES["channel"], math) for _ in range(2))
    unit = 0.5 * a.computeDt()
    dt = None if given is None else given(unit)
    for length in (unit * 230.3, unit * 0.1, 0.0, unit * 31, np.float32(unit * 2.5), 3 * unit):
        print("case simulate", scheme, math, length, flush=True)
        a.simulate(length, dt)
        step_loop(b, length, dt)
        assert a.simTime() == b.simTime() and type(a.simTime()) is type(b.simTime())
        assert a.simSteps() == b.simSteps() and a.computeDt() == b.computeDt() and a.dt == b.dt
        assert all(np.array_equal(x, y) for x, y in zip(a.download(), b.download()))
        for sim in (a, b):  # a substep pair changes the slots and buffers that the next run starts from
            sim.substep(np.float32(unit), 0)
            sim.substep(np.float32(unit), 1)
    assert a.simSteps() > 100


@pytest.mark.parametrize("scheme,math", [RUNS[0], RUNS[4]])
def test_simulate_calls_replaced_methods(ctx, scheme, math, monkeypatch):
    """A step or substep that a program wrapped is called for each step."""
    import functools

    sims = [make(ctx, scheme, state(scheme, 40, 30, seed=1), 40, 30, BOUNDARIES["reflective"], math)
            for _ in range(3)]
    cls = type(sims[0])
    calls = []
    dt = 0.1 * sims[0].computeDt()
    sims[0].simulate(dt * 7.5, dt)
    method = sims[1].step
    sims[1].step = lambda *a: (calls.append(0), method(*a))
    sims[1].simulate(dt * 7.5, dt)
    assert len(calls) == sims[0].simSteps() == sims[1].simSteps() == 8
    for name in ("step", "simTime"):
        calls.clear()
        inner = getattr(cls, name)
        monkeypatch.setattr(cls, name, functools.wraps(inner)(lambda *a: (calls.append(0), inner(*a))[1]))
        before = sims[2].simSteps()
        sims[2].simulate(dt * 7.5, dt)
        assert len(calls) >= sims[2].simSteps() - before >= 7
        monkeypatch.undo()
    assert all(np.array_equal(x, y) for x, y in zip(sims[0].download(), sims[1].download()))


def test_run_of_steps_refuses_bad_arguments(ctx):
    from finitevolumegpu_amd import _lib
    sim = make(ctx, "kp07_dimsplit", state("kp07_dimsplit", 40, 30, seed=1), 40, 30, BOUNDARIES["reflective"])
    out = sim._step_call.out_ptr
    sim._step_call._pack(sim, _lib.SCHEME_IDS["kp07_dimsplit"], 0.0, sim.boundary_conditions, sim.cfl_free)
    for kind, args, n in ((2, sim._step_call.args, out), (0, None, out), (0, sim._step_call.args, None)):
        with pytest.raises(_lib.FvmiError):
            _lib.call("fvmi_run_steps", kind, args, sim.launch, sim._step_call.time_ptr, 1.0, 0.1, 5, n, out, out,
                      sim.stream.handle)
    sim.nx = 1  # refused by the step, before anything is launched
    with pytest.raises(_lib.FvmiError):
        sim.simulate(0.1, 0.05)
    assert sim.simSteps() == 0 and sim.simTime() == 0.0


def _host_cfl(sim):
    h, hu, hv = (np.asarray(f, dtype=np.float64) for f in sim.download())
    c = np.sqrt(9.81 * h)
    return min((1.0 / (np.abs(hu / h) + c)).min(), (1.0 / (np.abs(hv / h) + c)).min())


@pytest.mark.parametrize("scheme,math", [("kp07_dimsplit", "fast"), ("hll2", "exact"), ("waf", "exact")])
@pytest.mark.parametrize("nx,ny", [(9, 8), (121, 33), (300, 251)])
def test_cfl_minimum_of_every_launch_shape(ctx, scheme, math, nx, ny):
    """The fastest cell, planted anywhere, gives the CFL minimum whichever wave
    of whichever workgroup holds it, in workgroups of one to four waves, the last
    of them partly without segments.  Bound: six roundings of 2^-23 (the sum,
    quotient, root and reciprocal, at most one unit each)."""
    rng = np.random.default_rng(nx)
    for waves, tile in ((1, 4), (2, 5), (3, 7), (4, 4), (4, 9), (4, 0)):
        h, hu, hv = (np.array(f) for f in state(scheme, nx, ny, seed=2))
        y, x = rng.integers(ny), rng.integers(nx)
        hv[y, x] = 6.0 * h[y, x]
        print("case cfl", scheme, math, nx, ny, waves, tile, (y, x), flush=True)
        sim = make(ctx, scheme, (h, hu, hv), nx, ny, BOUNDARIES["mixed"], math, waves_per_block=waves, tile_rows=tile)
        for _ in range(3):
            sim.step(np.float32(0.02))
            assert abs(sim.computeDt() / 0.5 / _host_cfl(sim) - 1.0) < 6 * 2.0 ** -23


@pytest.mark.parametrize("scheme", ["LxF", "HLL", "FORCE", "KP07"])
def test_unsplit_cfl_minimum_of_every_launch_shape(ctx, scheme):
    """Equal for every launch shape, one wave per workgroup included."""
    import importlib
    cls = getattr(importlib.import_module("finitevolumegpu_amd." + scheme), scheme)
    rng = np.random.default_rng(7)
    for nx, ny in ((9, 8), (121, 33), (300, 251)):
        h, hu, hv = (np.array(f) for f in state("kp07_dimsplit", nx, ny, seed=2))
        hv[rng.integers(ny), rng.integers(nx)] *= 40.0
        print("case unsplit cfl", scheme, nx, ny, flush=True)
        dts = set()
        for waves, tile in ((1, 4), (2, 5), (3, 7), (4, 4), (4, 9), (4, 0)):
            sim = cls(ctx, h, hu, hv, nx, ny, 1.0, 1.0, 9.81, waves_per_block=waves, tile_rows=tile)
            sim.step(np.float32(0.02))
            dts.add(sim.computeDt())
        assert len(dts) == 1 and 0.0 < dts.pop() < 1.0


@pytest.mark.parametrize("scheme,math", [("kp07_dimsplit", "fast"), ("ee2d_kp07_dimsplit", "fast"), ("kp07", "fast"),
                                         ("waf", "exact")])
@pytest.mark.parametrize("steps", [1, 2])
def test_recorded_steps_can_be_replayed(ctx, scheme, math, steps):
    """A graph of a program's own recording (one step: an odd number) goes on from
    its last replay, with eager work between."""
    import ctypes
    from finitevolumegpu_amd import _lib
    nx, ny = 61, 34
    fields = state(scheme, nx, ny, seed=5)
    a, b = (make(ctx, scheme, fields, nx, ny, BOUNDARIES["channel"], math) for _ in range(2))
    dt = np.float32(0.25 * a.computeDt())
    for sim in (a, b):
        sim.step(dt)
    print("case replay", scheme, math, flush=True)
    graph = ctypes.c_void_p()
    _lib.call("fvmi_stream_begin_capture", a.stream.handle)
    for _ in range(steps):
        a.step(dt)
    _lib.call("fvmi_stream_end_capture", a.stream.handle, ctypes.byref(graph))
    for _ in range(4):
        _lib.call("fvmi_graph_launch", graph, a.stream.handle)
        for _ in range(steps):
            b.step(dt)
        assert all(np.array_equal(x, y) for x, y in zip(a.download(), b.download()))
        assert a.computeDt() == b.computeDt()
    _lib.call("fvmi_graph_destroy", graph)
