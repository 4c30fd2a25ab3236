"""The square root of the exact arithmetic over the range of float32, as the CFL
minimum of still water shows it: 1 / sqrt(h) with g = dx = 1."""

import numpy as np
import pytest

from oracle import fv_oracle as O
from tests._cases import make_gpu_sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme,exponent", [("kp07_dimsplit", e) for e in (
    0, 1, 40, -50, -95, -96, -97, -101, -102, -112, -116, -120, -125, -126)] + [("waf", e) for e in (0, 1, -50)])
def test_square_root_of_the_exact_arithmetic(ctx, scheme, exponent):
    """Correctly rounded where the residuals that choose it are exact, that is
    multiples of 2^-149: from 2^-101 on.  Below, one unit from v_sqrt_f32, one from
    a residual that rounds to zero and half of one from the quotient."""
    n = 8
    rng = np.random.default_rng(exponent & 0xFF)
    mantissas = np.concatenate([[1.0, 1.0 + 2.0 ** -23, 2.0 - 2.0 ** -23], 1.0 + rng.random(9)])
    tolerance = 0.0 if exponent >= -101 else 2.5 * 2.0 ** -23
    print("case root", scheme, exponent, flush=True)
    for h in np.ldexp(mantissas, exponent).astype(np.float32):
        zero = np.zeros((n, n), dtype=np.float32)
        sim = make_gpu_sim(ctx, scheme, [zero + h, zero, zero], n, n, 1.0, 1.0, O.pack_bc(*[O.PERIODIC] * 4),
                           math="exact", g=1.0)
        sim.step(np.float32(0.0))
        want = np.float64(np.float32(1.0) / np.sqrt(h))
        assert abs(sim.computeDt() / 0.5 - want) <= tolerance * want, h
