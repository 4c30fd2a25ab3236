"""Where a simulator's state is between steps, as a program sees it: objects that
it holds, graphs that it recorded, ghost cells that it wrote and the table of an
ensemble.  Two simulators of the same state, one through whole steps and one
through its substeps, in which the state is back in its buffer after each step;
their results are equal."""

import ctypes

import numpy as np
import pytest

from oracle import fv_oracle as O
from tests._cases import make_gpu_sim, state
from tests.test_gpu_step import BOUNDARIES, make

pytestmark = pytest.mark.gpu

R, P, F, D = O.REFLECTIVE, O.PERIODIC, O.OUTFLOW, O.DIRICHLET

# one launch a step, and two
SCHEMES = [("kp07_dimsplit", "fast"), ("hll2", "fast"), ("ee2d_kp07_dimsplit", "fast"), ("kp07", "fast"),
           ("waf", "exact")]
DT = np.float32(2.0 ** -5)  # sums of a few are exact


def pair(ctx, scheme, math="fast", bc="channel", nx=61, ny=34):
    code = BOUNDARIES[bc] if isinstance(bc, str) else bc
    fields = state(scheme, nx, ny, seed=5)
    return [make(ctx, scheme, fields, nx, ny, code, math) for _ in range(2)]


def by_substeps(sim, steps=1):
    for _ in range(steps):
        for i in range(2):
            sim.substep(DT, i)


def assert_same(a, b):
    assert all(np.array_equal(x, y) for x, y in zip(a.download(), b.download()))
    assert a.computeDt() == b.computeDt()


@pytest.mark.parametrize("scheme,math", SCHEMES)
@pytest.mark.parametrize("steps", [1, 2, 3])
def test_held_state_stays_current(ctx, scheme, math, steps):
    a, b = pair(ctx, scheme, math)
    print("case held", scheme, math, steps, flush=True)
    out, fields = a.getOutput(), list(a.getOutput().gpu_variables)
    for advance in (lambda: [a.step(DT) for _ in range(steps)], lambda: a.simulate(float(steps * DT), DT)):
        advance()
        by_substeps(b, steps)
        assert a.getOutput() is out and all(x is y for x, y in zip(out.gpu_variables, fields))
        assert_same(a, b)
        assert all(np.array_equal(x, f.download(a.stream)) for x, f in zip(b.download(), fields))


def test_memory_outlives_the_simulator_with_either_field(ctx):
    """Both buffers of a variable live as long as one of its arrays, since a
    program's view of the array's memory may be of either."""
    import gc
    sim = pair(ctx, "kp07_dimsplit")[0]
    held = sim.u0[0]
    addresses = [held.data_ptr]
    sim.step(DT)
    addresses.append(held.data_ptr)
    state_now = sim.download()[0]
    sim.synchronize()
    del sim
    gc.collect()
    others = pair(ctx, "kp07_dimsplit")  # would be given freed memory
    assert not {x.data_ptr for s in others for u in (s.u0, s.u1) for x in u.gpu_variables} & set(addresses)
    assert np.array_equal(held.download(others[0].stream), state_now)


@pytest.mark.parametrize("scheme,math", SCHEMES)
def test_memory_goes_with_the_simulator(ctx, scheme, math):
    """Without the cycle collector, as large states are dropped in loops."""
    import gc
    import weakref
    gc.collect()
    gc.disable()
    try:
        sim = pair(ctx, scheme, math)[0]
        sim.step(DT)
        sim.simulate(float(DT), DT)
        sim.synchronize()
        memory = [weakref.ref(x.memory) for u in (sim.u0, sim.u1) for x in u.gpu_variables]
        held = sim.u0[0]
        del sim
        alive = [m() is not None for m in memory]
        assert sum(alive) == 2  # the held array's two
        del held
        assert all(m() is None for m in memory)
    finally:
        gc.enable()


def test_arrays_that_a_program_put_into_a_state(ctx):
    from finitevolumegpu_amd import Common
    a, b = pair(ctx, "kp07_dimsplit")
    a.step(DT)
    by_substeps(b)
    nx, ny = int(a.nx), int(a.ny)
    print("case own arrays", flush=True)
    a.u1 = Common.ArakawaA2D(a.stream, nx, ny, 2, 2, [None] * 3)
    own = a.u0.gpu_variables[1] = Common.HipArray2D(a.stream, nx, ny, 2, 2, a.download()[1])
    for _ in range(3):
        a.step(DT)
        by_substeps(b)
        assert a.u0[1] is own
        assert_same(a, b)


@pytest.mark.parametrize("scheme,math", SCHEMES)
@pytest.mark.parametrize("which", ["u0", "u1"])
def test_step_of_a_freed_array_is_refused(ctx, scheme, math, which):
    from finitevolumegpu_amd import _lib
    sim = pair(ctx, scheme, math)[0]
    sim.step(DT)
    sim.synchronize()
    print("case freed", scheme, math, which, flush=True)
    array = getattr(sim, which)[1]
    array.free()
    assert array.data_ptr is None
    with pytest.raises(_lib.FvmiError):
        sim.step(DT)
    with pytest.raises(_lib.FvmiError):
        sim.simulate(float(DT), DT)


def record(sim, enqueue):
    from finitevolumegpu_amd import _lib
    graph = ctypes.c_void_p()
    _lib.call("fvmi_stream_begin_capture", sim.stream.handle)
    try:
        enqueue()
    finally:
        _lib.call("fvmi_stream_end_capture", sim.stream.handle, ctypes.byref(graph))
    return graph


@pytest.mark.parametrize("how", ["step", "substep", "simulate"])
@pytest.mark.parametrize("scheme,math", SCHEMES)
def test_replays_and_eager_steps_in_turn(ctx, scheme, math, how):
    """A recorded step goes on from the latest state, whatever was stepped
    between its replays, and the other way round."""
    from finitevolumegpu_amd import _lib
    a, b = pair(ctx, scheme, math)
    a.step(DT)  # an odd number of steps before the recording
    by_substeps(b)
    print("case replays in turn", scheme, math, how, flush=True)
    graph = record(a, {"step": lambda: a.step(DT), "substep": lambda: by_substeps(a),
                       "simulate": lambda: a.simulate(float(DT), DT)}[how])
    for steps, run in ((1, 0), (0, 1), (0, 0), (3, 2), (2, 3), (1, 1)):
        _lib.call("fvmi_graph_launch", graph, a.stream.handle)
        by_substeps(b)
        assert_same(a, b)
        for _ in range(steps):
            a.step(DT)
        by_substeps(b, steps)
        assert_same(a, b)
        a.simulate(float(run * DT), DT)
        by_substeps(b, run)
        assert_same(a, b)
    _lib.call("fvmi_graph_destroy", graph)


@pytest.mark.parametrize("how", ["step", "exchange"])
@pytest.mark.parametrize("math", ["fast", "exact"])
def test_mpi_replays_and_eager_steps_in_turn(ctx, math, how):
    from finitevolumegpu_amd import _lib
    from finitevolumegpu_amd.MPISimulator import MPISimulator
    a, b = (MPISimulator(s) for s in pair(ctx, "ee2d_kp07_dimsplit", math))
    a.step(DT)
    by_substeps(b)
    print("case mpi replays", math, how, flush=True)
    graph = record(a, (lambda: a.step(DT)) if how == "step" else a.full_exchange)
    for steps in (1, 0, 3, 2):
        _lib.call("fvmi_graph_launch", graph, a.stream.handle)
        if how == "step":
            by_substeps(b)
        else:
            b.full_exchange()
        for _ in range(steps):
            a.step(DT)
        by_substeps(b, steps)
        assert_same(a, b)
        nx, ny = int(a.nx), int(a.ny)
        padded = [[v.download(s.stream, extent=[0, 0, nx + 4, ny + 4]) for v in s.getOutput().gpu_variables]
                  for s in (a, b)]
        assert all(np.array_equal(x, y) for x, y in zip(*padded))
    _lib.call("fvmi_graph_destroy", graph)


def write_ghosts(sim, seed):
    """Ghost cells of both buffers, others in each, around their interiors."""
    rng = np.random.default_rng(seed)
    ny, nx = sim.download()[0].shape
    for buf in (sim.u0, sim.u1):
        for k, v in enumerate(buf.gpu_variables):
            pad = (np.array([1.05, 0.01, -0.01, 6.5])[k] * rng.uniform(0.9, 1.1, (ny + 4, nx + 4))).astype(np.float32)
            pad[2:-2, 2:-2] = v.download(sim.stream)
            v.upload(sim.stream, pad, extent=[0, 0, nx + 4, ny + 4])


@pytest.mark.parametrize("math", ["fast", "exact"])
@pytest.mark.parametrize("edges", [(D, D, P, P), (P, P, D, R), (F, D, P, P)])
def test_mpi_step_with_a_dirichlet_edge(ctx, math, edges):
    """Beside an exchanged edge, the corners of a Dirichlet edge are memory that
    the exchange does not write."""
    from finitevolumegpu_amd.MPISimulator import MPISimulator
    sims = []
    for sim in pair(ctx, "ee2d_kp07_dimsplit", math, O.pack_bc(*edges)):
        write_ghosts(sim, seed=9)
        sims.append(MPISimulator(sim))
    print("case mpi dirichlet", math, edges, flush=True)
    for _ in range(3):
        sims[0].step(DT)
        by_substeps(sims[1])
        assert_same(*sims)


@pytest.mark.parametrize("scheme", ["kp07_dimsplit", "ee2d_kp07_dimsplit", "kp07"])
@pytest.mark.parametrize("before", [1, 2, 3])
def test_ghost_cells_written_before_a_dirichlet_edge(ctx, scheme, before):
    """A substep under Dirichlet edges reads the ghost cells that its input
    buffer was given, also those given while other edges were in force."""
    from finitevolumegpu_amd.Simulator import BoundaryCondition
    a, b = pair(ctx, scheme)
    print("case ghosts", scheme, before, flush=True)
    for sim in (a, b):
        write_ghosts(sim, seed=3)
    for _ in range(before):
        a.step(DT)
    by_substeps(b, before)
    for sim in (a, b):
        sim.setBoundaryConditions(BoundaryCondition(BoundaryCondition.getTypes(O.pack_bc(D, D, R, D))))
    for _ in range(3):
        a.step(DT)
        by_substeps(b)
        assert_same(a, b)


@pytest.mark.parametrize("steps", [1, 2])
def test_ensemble_after_replays_of_a_recorded_block(ctx, steps):
    """download() and nonfinite_counts() show the state after a program's own
    replays of a block that it recorded."""
    from finitevolumegpu_amd import _lib
    from finitevolumegpu_amd.Ensemble import Ensemble
    nx, ny = 57, 33
    fields = state("kp07_dimsplit", nx, ny, 3)
    spec = {"fields": fields, "nx": nx, "ny": ny, "dx": 1.0, "dy": 1.0, "g": 9.81, "t_end": 1e9,
            "bc": BOUNDARIES["reflective"], "dt": float(DT)}
    ens = Ensemble(ctx, "kp07_dimsplit", [spec], steps_per_graph=steps, use_graph=False)
    sim = make_gpu_sim(ctx, "kp07_dimsplit", fields, nx, ny, 1.0, 1.0, BOUNDARIES["reflective"])
    ens.advance()
    by_substeps(sim, steps)
    print("case ensemble replays", steps, flush=True)
    graph = record(ens, lambda: ens.advance(wait=False))
    for _ in range(3):
        _lib.call("fvmi_graph_launch", graph, ens.stream.handle)
        by_substeps(sim, steps)
        assert all(np.array_equal(x, y) for x, y in zip(ens.download(0), sim.download()))
    _lib.call("fvmi_graph_destroy", graph)
    ens.close()
