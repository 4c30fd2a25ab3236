"""The captured graph of an ensemble is destroyed only after the stream that may
still run it has been waited for.  On the CPU, with the library's calls recorded."""

import ctypes

import numpy as np
import pytest

from finitevolumegpu_amd import _lib
from finitevolumegpu_amd import Ensemble as module
from finitevolumegpu_amd.Simulator import BoundaryCondition

T = BoundaryCondition.Type
REFLECTIVE = int(BoundaryCondition.uniform(T.Reflective).asCodedInt())
DIRICHLET = int(BoundaryCondition.uniform(T.Dirichlet).asCodedInt())


class _Stream:
    handle = 0x51


class _Library:
    """Stands for the shared library: every call succeeds and is noted."""

    def __init__(self, log):
        self.log = log

    def __getattr__(self, name):
        return lambda *args: (self.log.append(name), 0)[1]


@pytest.fixture
def running(monkeypatch):
    """A two-slot ensemble with a graph in flight, and the log of calls."""
    log = []
    monkeypatch.setattr(_lib, "call", lambda name, *args: (log.append(name), 0)[1])
    monkeypatch.setattr(_lib, "_lib", _Library(log))
    _Stream.synchronize = lambda self: log.append("synchronize")
    ens = object.__new__(module.Ensemble)
    ens.scheme, ens.math, ens.seg_rows, ens.min_seg_rows = "kp07_dimsplit", "fast", None, 24
    ens.n, ens.stream, ens.graph, ens._host_refs = 2, _Stream(), ctypes.c_void_p(0x71), []
    ens.host_table = (_lib.Instance * 2)()
    ens.tab = np.frombuffer(ens.host_table, dtype=_lib.INSTANCE_DTYPE)
    ens.table = ctypes.c_void_p(0x72)
    ens.live = np.array([True, False])
    ens.tab["nx"], ens.tab["ny"] = 64, 64
    ens.arena, ens.own_arena, ens.buffers = None, False, [None, None]
    yield ens, log
    ens.graph = None
    del ens.stream


@pytest.mark.parametrize("whole,bc", [(False, REFLECTIVE), (True, DIRICHLET)])
def test_turning_between_substeps_and_whole_steps(running, whole, bc):
    ens, log = running
    ens.whole_steps = whole
    ens.tab["bc"] = bc
    ens._choose_steps()
    assert ens.whole_steps is not whole and ens.graph is None
    assert "synchronize" in log[:log.index("fvmi_graph_destroy")]


def test_close_waits_for_the_graph(running):
    ens, log = running
    ens.close()
    assert "synchronize" in log[:log.index("fvmi_graph_destroy")]
