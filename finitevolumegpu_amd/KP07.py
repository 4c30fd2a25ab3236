"""Unsplit second-order Kurganov-Petrova shallow-water scheme with TVD
Runge-Kutta time stepping (GPUSimulators/KP07.py; kernel
GPUSimulators/cuda/SWE2D_KP07.cu)."""

import operator

import numpy as np

from . import _lib
from .Simulator import BoundaryCondition, UnsplitSimulator, _StepCall, _steps_in_library, swe_initial_cfl


def stepOrderToCodedInt(step, order):
    """Simulator.stepOrderToCodedInt: step << 16 | order."""
    return (int(step) << 16) | (int(order) & 0xFFFF)


class KP07(UnsplitSimulator):
    """Constructor signature of KP07.__init__ (KP07.py:54-106): ``order`` RK
    stages per step (1 or 2), computeDt = min(cfl) * 0.5**(order-1)."""

    scheme = "kp07"
    gc = 2
    nvars = 3
    _substep_names = ("substep", "_launch", "_field_args", "cfl_pointer")
    _methods_of = operator.attrgetter(*_substep_names)

    def __init__(self, context, h0, hu0, hv0, nx, ny, dx, dy, g, theta=1.3, cfl_scale=0.9, order=2,
                 boundary_conditions=BoundaryCondition(), block_width=16, block_height=16,
                 tile_rows=None, waves_per_block=None, math=None, xcd_remap=True):
        if order not in (1, 2):
            raise ValueError("order must be 1 or 2")
        super().__init__(context, nx, ny, dx, dy, boundary_conditions, cfl_scale, order, block_width, block_height)
        self.g = np.float32(g)
        self.theta = np.float32(theta)
        self.order = order
        self.dt_factor = 0.5 ** (order - 1)
        self._init_unsplit([h0, hu0, hv0], swe_initial_cfl(h0, hu0, hv0, self.dx, self.dy, g),
                           tile_rows, waves_per_block, math, xcd_remap)
        # a second-order step is one library call
        self._step_call = _StepCall("fvmi_swe_kp07_rk2_step", _lib.RUN_KP07_RK2)
        if order == 2:
            self._find_own_methods()

    def step(self, dt):
        """One full step; with two stages as one library call
        (fvmi_swe_kp07_rk2_step) with the results of the two substeps."""
        if not self._one_call():
            super().step(dt)
            return
        self._take_step(*self._step_call.step(self, 0, np.float32(dt), self.boundary_conditions, 1 - self.cfl_last))
        self.t += float(dt)
        self.nt += 1

    def _take_step(self, in_other, slot):
        if in_other:
            self.pair.turn.value ^= 1
        elif self.math == "fast":
            self._note_recording()
        self.cfl_last = slot

    def _run_steps(self, t_end, max_steps):
        self._note_recording()
        return (self._one_call() and _steps_in_library(self)
                and self._step_call.run(self, 0, t_end, max_steps, 1 - self.cfl_last))

    def substep(self, dt, step_number):
        self._note_recording()
        super().substep(dt, step_number)

    def substepRK(self, dt, substep):
        self.substep(dt, substep)

    def _launch(self, dt, substep, u0, u1, cfl, slot):
        _lib.call("fvmi_swe_kp07_substep", int(self.nx), int(self.ny), float(self.dx), float(self.dy), float(dt),
                  float(self.g), float(self.theta), stepOrderToCodedInt(substep, self.order),
                  int(self.boundary_conditions), *self._field_args(u0), *self._field_args(u1), cfl, slot,
                  self.launch, self.stream.handle)
