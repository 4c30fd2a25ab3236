"""NaN, infinities, zero and negative depths in the whole-step and Runge-Kutta
launches: the fields and the CFL minimum of the two substep launches, NaN where they
have NaN, and nothing else than they have anywhere."""

import numpy as np
import pytest

from tests._cases import state
from tests.test_gpu_step import BOUNDARIES, make

pytestmark = pytest.mark.gpu

SCHEMES = ["kp07_dimsplit", "hll2", "ee2d_kp07_dimsplit", "kp07"]
VALUES = {"nan": np.nan, "inf": np.inf, "-inf": -np.inf, "zero": 0.0, "negative": -1.0, "lowest": -3.4e38}


@pytest.mark.parametrize("value", sorted(VALUES))
@pytest.mark.parametrize("scheme", SCHEMES)
def test_step_equals_its_substeps_around_special_values(ctx, scheme, value):
    nx, ny = 130, 61
    for bc in ("reflective", "periodic", "mixed", "channel"):
        # in the middle of a strip, at its edges, in corners and on ghost rows' sources
        for y, x in ((30, 70), (0, 0), (ny - 1, nx - 1), (1, 56), (ny - 2, 55), (29, 112), (30, 1)):
            print("case special", scheme, value, bc, y, x, flush=True)
            fields = [f.copy() for f in state(scheme, nx, ny, seed=6)]
            fields[(x + y) % len(fields)][y, x] = VALUES[value]
            with np.errstate(all="ignore"):
                a, b = (make(ctx, scheme, fields, nx, ny, BOUNDARIES[bc]) for _ in range(2))
            dt = np.float32(0.04)
            for _ in range(2):
                a.step(dt)
                for i in range(2):
                    b.substep(dt, i)
                for k, (p, q) in enumerate(zip(a.download(), b.download())):
                    assert np.array_equal(p, q, equal_nan=True), (k, np.argwhere(p != q)[:5].tolist())
                assert np.array_equal(a.computeDt(), b.computeDt(), equal_nan=True)
