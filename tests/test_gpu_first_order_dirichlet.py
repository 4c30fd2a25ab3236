"""One-ghost-cell schemes with two columns per lane at Dirichlet edges, whose first
strip reads from the ghost column on: equal to one column per lane, and the ghost
cells untouched."""

import importlib

import numpy as np
import pytest

from oracle import fv_oracle as O
from tests._cases import state

pytestmark = pytest.mark.gpu

R, P, F, D = O.REFLECTIVE, O.PERIODIC, O.OUTFLOW, O.DIRICHLET


@pytest.mark.parametrize("scheme", ["LxF", "HLL", "FORCE"])
@pytest.mark.parametrize("edges", [(D, D, D, D), (R, F, D, D), (R, R, R, D), (P, P, D, F), (D, R, F, R)])
def test_two_columns_per_lane_at_dirichlet_edges(ctx, scheme, edges):
    """One-row segments make enough waves for two columns per lane, 64-row segments
    leave one; edges in the order north, south, east, west."""
    from finitevolumegpu_amd.Simulator import BoundaryCondition
    cls = getattr(importlib.import_module("finitevolumegpu_amd." + scheme), scheme)
    bc = BoundaryCondition(dict(zip(("north", "south", "east", "west"), edges)))
    ny = 1100
    for nx in (2, 3, 123, 124, 125, 247, 250):
        print("case dirichlet columns", scheme, edges, nx, flush=True)
        rng = np.random.default_rng(nx)
        padded = []
        for k, f in enumerate(state("kp07_dimsplit", nx, ny, seed=nx)):
            pad = ((1.05, 0.02, -0.03)[k] * rng.uniform(0.9, 1.1, (ny + 2, nx + 2))).astype(np.float32)
            pad[1:-1, 1:-1] = f
            padded.append(pad)
        sims = [cls(ctx, *[p[1:-1, 1:-1].copy() for p in padded], nx, ny, 1.0, 1.0, 9.81, boundary_conditions=bc,
                    tile_rows=rows) for rows in (1, 64)]
        for sim in sims:
            for buf in (sim.u0, sim.u1):
                for k, pad in enumerate(padded):
                    buf[k].upload(sim.stream, pad, extent=[0, 0, nx + 2, ny + 2])
        dt = np.float32(0.1)
        for _ in range(3):
            for sim in sims:
                sim.step(dt)
        assert all(np.array_equal(x, y) for x, y in zip(*[s.download() for s in sims])), nx
        assert sims[0].computeDt() == sims[1].computeDt()
        for k, pad in enumerate(padded):
            got = sims[0].u0[k].download(sims[0].stream, extent=[0, 0, nx + 2, ny + 2])
            got[1:-1, 1:-1] = pad[1:-1, 1:-1]
            assert np.array_equal(got, pad)
