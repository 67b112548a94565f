"""SCABit MCS captured into a graph on the scheduler's stream: the graph holds
half-sweeps of the lattice itself, not the spare lattice of the one-pass MCS,
which the scheduler may give back before the graph is replayed."""
import ctypes as C

import numpy as np
import pytest

import cudakpz_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu

RELAXED = 2  # hipStreamCaptureModeRelaxed


class Graph:
    """What `work()` queues on the stream, as an executable graph."""

    def __init__(self, stream, work):
        self.h = C.CDLL("libamdhip64.so")
        self.stream, self.graph, self.exe = C.c_void_p(stream), C.c_void_p(), C.c_void_p()
        assert self.h.hipStreamBeginCapture(self.stream, RELAXED) == 0
        work()
        assert self.h.hipStreamEndCapture(self.stream, C.byref(self.graph)) == 0
        assert self.h.hipGraphInstantiate(C.byref(self.exe), self.graph, None, None, C.c_size_t(0)) == 0

    def nodes(self):
        n = C.c_size_t()
        assert self.h.hipGraphGetNodes(self.graph, None, C.byref(n)) == 0
        return n.value

    def replay(self):
        assert self.h.hipGraphLaunch(self.exe, self.stream) == 0

    def close(self):
        assert self.h.hipGraphExecDestroy(self.exe) == 0
        assert self.h.hipGraphDestroy(self.graph) == 0


@pytest.mark.parametrize("lx,ly,T", [(9, 7, 0), (14, 6, 7), (15, 6, 0)])
def test_captured_mcs(lx, ly, T):
    s = K.SchedulerSCABit(lx, ly, threads=T)
    s.supplySeed(8)
    s.initHomogeneous()
    s.mcs(2)  # tables, and the spare lattice
    s.sync()
    g = Graph(s.stream, lambda: s.mcs(4))
    assert g.nodes() == 8  # 4 MCS, two half-sweeps each
    n = 2
    m = O.Dsfmt(O.seed32(8))
    st = O.Streams(s.threads, m)
    lat = O.flat(lx, ly, O.ENC_CBBIT)
    O.cbbit_mcs(lat, lx, ly, st, 2, 0)
    for eager in (0, 2, 1, 3):
        K.releaseSpares()
        g.replay()
        s.mcs(eager)  # the program's own steps between the replays
        s.sync()
        O.cbbit_mcs(lat, lx, ly, st, 4 + eager, 0)
        assert np.array_equal(s.popSystem(), lat)
        assert np.array_equal(s.streams(), st.states)
    g.close()
