"""Long and narrow lattices on the rules that choose kernels by shape: results
against the oracle on both sides of each line, and times that may not fall off
where a kernel is the wrong one for a shape."""
import os
import time

import numpy as np
import pytest

import cudakpz_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu

THREADS = max(1, min(16, os.cpu_count() or 1))
CLS = {O.ENC_LOCAL: K.SchedulerDT, O.ENC_CBBIT: K.SchedulerSCABit}


def random_lattice(s, seed):
    return np.random.default_rng(seed).integers(0, 1 << 32, s.size_words, dtype=np.uint64).astype(np.uint32)


def seconds(s, f):
    """shortest of several runs of f, waited for"""
    best = np.inf
    for _ in range(7):
        s.sync()
        t = time.perf_counter()
        f()
        s.sync()
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("enc,lx,ly", [(O.ENC_LOCAL, 5, 14), (O.ENC_LOCAL, 5, 15), (O.ENC_LOCAL, 7, 13), (O.ENC_LOCAL, 7, 14),
                                       (O.ENC_LOCAL, 15, 5), (O.ENC_LOCAL, 16, 5), (O.ENC_LOCAL, 16, 6),
                                       (O.ENC_CBBIT, 6, 13), (O.ENC_CBBIT, 6, 14), (O.ENC_CBBIT, 7, 14), (O.ENC_CBBIT, 7, 15),
                                       (O.ENC_CBBIT, 8, 16), (O.ENC_CBBIT, 14, 5), (O.ENC_CBBIT, 15, 5)])
def test_correlate(enc, lx, ly):
    s = CLS[enc](lx, ly)
    snap, lat = random_lattice(s, 1), random_lattice(s, 2)
    s.pushSystem(snap)
    s.correlateTag()
    s.pushSystem(lat)
    c = s.correlate()
    assert (c.sum_h, c.sum_hs, c.sum_h2, c.sum_hhs, c.tcs) == O.correlate_rows(lat, snap, enc, lx, ly, THREADS)


def correlate_time(cls, lx, ly):
    s = cls(lx, ly)
    s.initHomogeneous()
    s.correlateTag()
    return seconds(s, s.correlate)


def test_correlate_time():
    # a quarter of the rows; with a wave for each of 2^17 narrow rows 0.64, by tables 0.31
    assert correlate_time(K.SchedulerDT, 7, 17) < 0.5 * correlate_time(K.SchedulerDT, 7, 19)
    # 64 rows against 128; with one wave for each long row 1.8, by tables 1.0
    assert correlate_time(K.SchedulerSCABit, 18, 6) < 1.3 * correlate_time(K.SchedulerSCABit, 18, 7)


# 2^12 word rows of four site rows, one for each workgroup, and twice to eight times as many
@pytest.mark.parametrize("ly", [14, 15, 17])
def test_moments_of_many_rows(ly):
    s = K.SchedulerDT(6, ly)
    lat = random_lattice(s, ly)
    s.pushSystem(lat)
    got = s.moments()
    h = O.heights(lat, O.ENC_LOCAL, 6, ly).astype(np.int64).ravel()
    values, counts = np.unique(h, return_counts=True)
    for k in range(1, 8):
        exact = sum(int(v) ** k * int(c) for v, c in zip(values, counts))
        size = sum(abs(int(v)) ** k * int(c) for v, c in zip(values, counts))
        # some ten roundings per site and level of the sums, each half an ulp of the absolute sum
        assert abs(got[k - 1] * h.size - exact) <= 2.0 ** -52 * 16 * size


def test_moments_time():
    # 64 rows of 2^18 sites against a square of as many: 13 times as long with
    # one wave for four of the long rows, 6 with a wave each
    s, t = K.SchedulerDT(18, 6), K.SchedulerDT(12, 12)
    s.initHomogeneous()
    t.initHomogeneous()
    assert seconds(s, s.moments) < 10 * seconds(t, t.moments)


# rows of 1 to 8 words on tall lattices: one pass in bands of 2 rows up to 2^26
# sites, half-sweeps above; rows of 8 words in one pass throughout
@pytest.mark.parametrize("lx,ly,T", [(7, 19, 0), (8, 18, 1000), (9, 17, 0), (9, 18, 7), (10, 17, 1000)])
def test_tall_scabit(lx, ly, T):
    s = K.SchedulerSCABit(lx, ly, threads=T)
    s.supplySeed(12)
    s.initHomogeneous()
    s.mcs(2)
    s.mcs(3)
    m = O.Dsfmt(O.seed32(12))
    st = O.Streams(s.threads, m)
    lat = O.flat(lx, ly, O.ENC_CBBIT)
    O.cbbit_mcs_threaded(lat, lx, ly, st, 5, 0, 0.5, 0.0, THREADS)
    assert np.array_equal(s.popSystem(), lat)
    assert np.array_equal(s.streams(), st.states)


@pytest.mark.parametrize("lx,ly", [(7, 22), (8, 18), (8, 20), (9, 18), (10, 20)])
def test_tall_scabit_time(lx, ly):
    # ten MCS in one call against ten calls of one, which are half-sweeps
    # (3 to 6 times as long on rows of 1 and 2 words with bands of 16 and more rows)
    s = K.SchedulerSCABit(lx, ly)
    s.initHomogeneous()
    s.mcs(2)
    assert seconds(s, lambda: s.mcs(10)) < 1.2 * seconds(s, lambda: [s.mcs(1) for _ in range(10)])
