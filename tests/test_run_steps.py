"""Between two progress reports of simulate() lies little work for the device: a
library call takes few steps of a large grid, and up to 100 of a small one."""

from types import SimpleNamespace

import numpy as np
import pytest

from finitevolumegpu_amd import _lib
from finitevolumegpu_amd.Simulator import _StepCall


@pytest.mark.parametrize("nx,ny", [(128, 128), (700, 900), (1024, 1024), (4096, 4096), (16000, 16000)])
def test_steps_of_one_library_call(monkeypatch, nx, ny):
    asked = []
    monkeypatch.setattr(_lib, "call", lambda name, *args: asked.append(args[6]))
    state = SimpleNamespace(gpu_variables=[])
    pair = SimpleNamespace(places_of=lambda u, v: (0,) * 16)
    sim = SimpleNamespace(nx=np.int32(nx), ny=np.int32(ny), dx=1.0, dy=1.0, g=9.81, u0=state, u1=state, pair=pair, t=0.0,
                          dt=0.5, boundary_conditions=0, cfl_pointer=lambda: 0, launch=None,
                          stream=SimpleNamespace(handle=None))
    for left in (100, 7, 1):
        _StepCall("fvmi_dimsplit_step", _lib.RUN_DIMSPLIT).run(sim, 0, 1e9, left, 0)
    assert all(1 <= n <= left for n, left in zip(asked, (100, 7, 1)))
    # 2^27 cells are less than 2 ms of work
    assert asked[0] == 1 or asked[0] * nx * ny <= 2 ** 27
    assert asked[0] == 100 or (asked[0] + 1) * nx * ny > 2 ** 27
