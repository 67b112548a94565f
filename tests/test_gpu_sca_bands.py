"""SchedulerSCA against the oracle with every band height of its kernel (2 to
64 cell rows, chosen by the lattice size) and with few and many worker streams."""
import os

import numpy as np
import pytest

import cudakpz_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu

THREADS = max(1, min(16, os.cpu_count() or 1))


# sites 2^20: bands of 2 rows; 2^22 .. 2^24: 4; then 8, 16, 32, 64.  The last
# two of 2 and 4 rows: a single band row, and one group of columns per row
@pytest.mark.parametrize("lx,ly", [(10, 10), (12, 10), (13, 11), (13, 13), (14, 13), (14, 14), (15, 14), (14, 3), (17, 4),
                                   (8, 14)])
@pytest.mark.parametrize("T", [0, 37])
def test_band_heights(lx, ly, T):
    s = K.SchedulerSCA(lx, ly, threads=T)
    s.supplySeed(19)
    s.initHomogeneous()
    s.setPQ(0.9, 0.2)
    s.mcsPQSyncRng(2)
    m = O.Dsfmt(O.seed32(19))
    st = O.Streams(s.threads, m)
    lat = O.flat(lx, ly, O.ENC_LOCAL)
    O.cb_mcs_threaded(lat, lx, ly, st, 2, 0.9, 0.2, THREADS)
    assert np.array_equal(s.popSystem(), lat)
    assert np.array_equal(s.streams(), st.states)
