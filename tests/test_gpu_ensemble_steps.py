"""Ensembles that take whole steps in one launch: Euler instances, and turning
between whole steps and substeps while blocks are in flight.  Every instance equals
its plain run."""

import numpy as np
import pytest

from oracle import fv_oracle as O
from tests._cases import state
from tests.test_gpu_step import BOUNDARIES, make

pytestmark = pytest.mark.gpu

R, P, F, D = O.REFLECTIVE, O.PERIODIC, O.OUTFLOW, O.DIRICHLET


def spec_of(scheme, nx, ny, bc, t_end, seed):
    euler = scheme == "ee2d_kp07_dimsplit"
    spec = {"fields": state(scheme, nx, ny, seed), "nx": nx, "ny": ny, "dx": 1.0, "dy": 1.0,
            "g": 0.1 if euler else 9.81, "t_end": t_end, "bc": bc}
    if euler:
        spec["gamma"] = 1.4
    return spec


def assert_plain_run(ctx, ens, i, scheme, spec):
    sim = make(ctx, scheme, spec["fields"], spec["nx"], spec["ny"], spec["bc"])
    sim.simulate(spec["t_end"])
    assert ens.state(i) == (sim.simTime(), sim.simSteps()), i
    assert all(np.array_equal(x, y) for x, y in zip(ens.download(i), sim.download())), i
    return sim.simSteps()


@pytest.mark.parametrize("steps_per_graph,seg_rows", [(1, None), (3, None), (4, 5)])
def test_euler_instances(ctx, steps_per_graph, seg_rows):
    from finitevolumegpu_amd.Ensemble import Ensemble
    scheme = "ee2d_kp07_dimsplit"
    edges = ("reflective", "mixed", "periodic", "outflow", "channel", "reflective")
    sizes = [(8, 8), (57, 33), (113, 65), (70, 120), (56, 9), (300, 47)]
    specs = [spec_of(scheme, nx, ny, BOUNDARIES[k], 1.1 + 0.37 * j, 30 + j)
             for j, ((nx, ny), k) in enumerate(zip(sizes, edges))]
    print("case euler instances", steps_per_graph, seg_rows, flush=True)
    ens = Ensemble(ctx, scheme, specs, math="fast", steps_per_graph=steps_per_graph, seg_rows=seg_rows)
    ens.run()
    assert ens.whole_steps
    assert {assert_plain_run(ctx, ens, i, scheme, s) % 2 for i, s in enumerate(specs)} == {0, 1}
    assert (ens.nonfinite_counts(range(len(specs))) == 0).all()
    ens.close()


@pytest.mark.parametrize("late", [O.pack_bc(D, R, D, R), O.pack_bc(R, R, P, R)])
@pytest.mark.parametrize("scheme", ["kp07_dimsplit", "ee2d_kp07_dimsplit"])
def test_turning_both_ways_without_waiting(ctx, scheme, late):
    """An instance that needs substeps joins between blocks and leaves again, and
    the next one turns the ensemble back to whole steps with a block in flight."""
    from finitevolumegpu_amd.Ensemble import Ensemble
    specs = [spec_of(scheme, 57, 33, BOUNDARIES["reflective"], 6.0, 1),
             spec_of(scheme, 90, 64, BOUNDARIES["periodic"], 7.3, 2)]
    guest = spec_of(scheme, 40, 30, late, 1.0, 3)
    # Dirichlet edges read the instance's ghost memory, which is zero: keep it out of the
    # comparison and only in the company of the others
    print("case turning", scheme, late, flush=True)
    ens = Ensemble(ctx, scheme, specs, math="fast", steps_per_graph=3, capacity=4)
    ens.advance(wait=False)
    assert ens.whole_steps
    slot = ens.add(guest)
    ens.advance(wait=False)
    ens.advance(wait=False)
    assert not ens.whole_steps
    while slot not in ens.finished():
        ens.advance()
    ens.advance()  # a plan without the guest
    ens.plan(ens._active_mask())
    ens.remove(slot)
    ens.advance(wait=False)
    specs.append(spec_of(scheme, 64, 48, BOUNDARIES["outflow"], 2.0, 4))
    third = ens.add(specs[2])
    ens.advance(wait=False)
    assert ens.whole_steps
    ens.run()
    for i, s in zip((0, 1, third), specs):
        assert_plain_run(ctx, ens, i, scheme, s)
    ens.close()
