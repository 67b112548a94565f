"""Bit-parallel SCABit MCS in one pass (two or more MCS in a call) against the
oracle: every row width class of the kernel (up to 64 words, 128, more), bands
from 2 rows on, odd and even numbers of MCS, workers with one, several and uneven
numbers of rows."""
import os

import numpy as np
import pytest

import cudakpz_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu

THREADS = max(1, min(16, os.cpu_count() or 1))


def run(lx, ly, T, calls):
    s = K.SchedulerSCABit(lx, ly, threads=T)
    s.supplySeed(23)
    s.initHomogeneous()
    for n in calls:
        s.mcs(n)
    m = O.Dsfmt(O.seed32(23))
    st = O.Streams(s.threads, m)
    lat = O.flat(lx, ly, O.ENC_CBBIT)
    O.cbbit_mcs_threaded(lat, lx, ly, st, sum(calls), 0, 0.5, 0.0, THREADS)
    assert np.array_equal(s.popSystem(), lat)
    assert np.array_equal(s.streams(), st.states)
    assert s.mcsCount() == sum(calls)
    ptr = s.device_lattice
    s.mcs(2)
    assert s.device_lattice == ptr


@pytest.mark.parametrize("lx", [7, 8, 12, 13, 14, 15, 16, 18])
@pytest.mark.parametrize("ly,T", [(2, 0), (2, 3), (5, 0), (6, 7), (7, 1)])
def test_row_widths(lx, ly, T):
    run(lx, ly, T, (3, 2))


# bands of 2 to 64 rows
@pytest.mark.parametrize("lx,ly,T", [(9, 9, 0), (7, 13, 100), (11, 14, 0), (14, 12, 0), (14, 13, 1000), (15, 13, 0),
                                     (13, 15, 0), (16, 13, 37), (18, 11, 0)])
def test_bands(lx, ly, T):
    run(lx, ly, T, (2, 1, 4))


def test_pq_at_half():
    # p = .5, q = 0 through the p/q call takes the same path; another (p, q) in between does not
    s = K.SchedulerSCABit(15, 6)
    s.supplySeed(4)
    s.initHomogeneous()
    s.setPQ(0.5, 0.0)
    s.mcsPQSyncRng(4)
    s.setPQ(0.9, 0.1)
    s.mcsPQSyncRng(3)
    s.mcs(2)
    m = O.Dsfmt(O.seed32(4))
    st = O.Streams(s.threads, m)
    lat = O.flat(15, 6, O.ENC_CBBIT)
    O.cbbit_mcs(lat, 15, 6, st, 4, 0)
    O.cbbit_mcs(lat, 15, 6, st, 3, 1, 0.9, 0.1)
    O.cbbit_mcs(lat, 15, 6, st, 2, 0)
    assert np.array_equal(s.popSystem(), lat)
    assert np.array_equal(s.streams(), st.states)


# the per-site rule takes one pass from 2^31 sites on (512 MiB)
@pytest.mark.parametrize("lx,ly,T,p,q", [(18, 13, 37, 0.7, 0.0), (15, 16, 0, 0.95, 0.05)])
def test_per_site_in_one_pass(lx, ly, T, p, q):
    s = K.SchedulerSCABit(lx, ly, threads=T)
    s.supplySeed(31)
    s.initHomogeneous()
    s.setPQ(p, q)
    s.mcsPQSyncRng(3)
    m = O.Dsfmt(O.seed32(31))
    st = O.Streams(s.threads, m)
    lat = O.flat(lx, ly, O.ENC_CBBIT)
    O.cbbit_mcs_threaded(lat, lx, ly, st, 3, 1, p, q, THREADS)
    assert np.array_equal(s.popSystem(), lat)
    assert np.array_equal(s.streams(), st.states)
