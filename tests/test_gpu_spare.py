"""The spare lattice of SCABit's one-pass MCS is memory that other allocations
find as if it were free: a failing allocation of the library takes it back, and
the scheduler goes on with half-sweeps or another spare, with the same results."""
import ctypes as C
import threading

import numpy as np
import pytest

import cudakpz_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu

GiB = 1 << 30


class Filled:
    """Device memory taken up to `left` bytes."""

    def __init__(self, left):
        self.h = C.CDLL("libamdhip64.so")
        self.h.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.h.hipFree.argtypes = [C.c_void_p]
        self.blocks = []
        while self.free() > left + GiB // 4:
            p = C.c_void_p()
            assert self.h.hipMalloc(C.byref(p), min(16 * GiB, self.free() - left)) == 0
            self.blocks.append(p)

    def free(self):
        free, total = C.c_size_t(), C.c_size_t()
        assert self.h.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for p in self.blocks:
            self.h.hipFree(p)


def seeded(lx, ly, seed, **kw):
    s = K.SchedulerSCABit(lx, ly, **kw)
    s.supplySeed(seed)
    s.initHomogeneous()
    return s


def sums(s):
    r = s.roughness()
    return r.sum_h, r.sum_h2


# each of them needs 4 GiB of its own
NEEDS = {
    "scheduler": lambda s: K.SchedulerSCABit(17, 17),
    "tag": lambda s: s.correlateTag(),
    "batch": lambda s: K.Batch([(K.KPZ_SCABIT, 17, 17, 0.5, 0.0, 1)]),
    "server": lambda s: K.Server(hbm_budget=4 * GiB, max_slots=1, max_tick_mcs=1),
}


@pytest.mark.parametrize("what", NEEDS)
def test_other_allocations_find_the_room(what):
    s = seeded(17, 17, 3)
    s.mcs(2)  # 4 GiB lattice, 4 GiB spare
    s.sync()
    with Filled(3 * GiB):
        other = NEEDS[what](s)
        s.mcs(3)
        got = sums(s)
        del other
    s.close()
    t = seeded(17, 17, 3)
    for _ in range(5):
        t.mcs(1)  # half-sweeps
    assert got == sums(t)
    t.close()


@pytest.mark.parametrize("lx,ly,T", [(8, 7, 0), (14, 6, 7), (16, 5, 0)])
def test_given_back_between_calls(lx, ly, T):
    s = seeded(lx, ly, 5, threads=T)
    m = O.Dsfmt(O.seed32(5))
    st = O.Streams(s.threads, m)
    lat = O.flat(lx, ly, O.ENC_CBBIT)
    for n in (4, 3, 1, 2):
        s.mcs(n)
        K.releaseSpares()
        O.cbbit_mcs(lat, lx, ly, st, n, 0)
    assert np.array_equal(s.popSystem(), lat)
    assert np.array_equal(s.streams(), st.states)
    s.mcs(2)
    assert K.releaseSpares() >= 4 * s.size_words
    assert K.releaseSpares() == 0


def test_both_rules_after_a_new_spare():
    # 2^31 sites: both rules take one pass, each with its own table behind the spare lattice
    s, t = seeded(17, 14, 9), seeded(17, 14, 9)
    for k in range(3):
        for p, q in ((0.5, 0.0), (0.9, 0.2)):
            for x, steps in ((s, (2,)), (t, (1, 1))):
                x.setPQ(p, q)
                for n in steps:
                    x.mcsPQSyncRng(n)
        assert K.releaseSpares() >= 4 * s.size_words if k != 1 else True
    assert sums(s) == sums(t)
    assert np.array_equal(s.streams(), t.streams())


def test_single_steps_take_no_spare():
    s = seeded(15, 15, 2)
    K.releaseSpares()
    for _ in range(3):
        s.mcs(1)
    assert K.releaseSpares() == 0
    s.mcs(3)
    assert K.releaseSpares() >= 4 * s.size_words


def test_given_back_by_another_thread():
    lx, ly, n = 12, 9, 600
    s = seeded(lx, ly, 6)
    ended = threading.Event()

    def steps():
        for _ in range(n // 2):
            s.mcs(2)
        s.sync()
        ended.set()

    t = threading.Thread(target=steps)
    t.start()
    while not ended.is_set():
        K.releaseSpares()
    t.join()
    m = O.Dsfmt(O.seed32(6))
    st = O.Streams(s.threads, m)
    lat = O.flat(lx, ly, O.ENC_CBBIT)
    O.cbbit_mcs_threaded(lat, lx, ly, st, n, 0, 0.5, 0.0, 8)
    assert np.array_equal(s.popSystem(), lat)
    assert np.array_equal(s.streams(), st.states)


# what bench.py accounts the memory by: the width and size limits of the rule,
# a row wider than the one-pass kernel takes, a spare that is not to be had
@pytest.mark.parametrize("lx,ly,rule,one", [(6, 9, "mcs", False), (7, 9, "mcs", True), (18, 5, "mcs", True), (19, 5, "mcs", False),
                                            (12, 12, "pq", False), (14, 17, "pq", False), (15, 16, "pq", True)])
def test_one_pass_is_told(lx, ly, rule, one):
    s = seeded(lx, ly, 1)
    s.setPQ(0.9, 0.1)
    advance = s.mcs if rule == "mcs" else s.mcsPQSyncRng
    advance(2)
    assert s.onePass() is one
    advance(1)
    assert s.onePass() is False
    assert K.SchedulerDT(8, 8).onePass() is False


def test_no_spare_is_told():
    s = seeded(18, 16, 1)  # 4 GiB: as large as a spare may be
    s.mcs(2)
    assert s.onePass()
    t = seeded(18, 17, 1)  # 8 GiB
    t.mcs(2)
    assert not t.onePass()
