"""The kernels a double-tiling phase can take, against the oracle at the sizes
where one hands over to the other: the p/q loop that draws in runs (from 2^18
blocks on).  Everything is compared word for word."""
import os

import numpy as np
import pytest

import cudakpz_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu

THREADS = max(1, min(16, os.cpu_count() or 1))
RULES = {"kpz": O.UPD_KPZ, "pq": O.UPD_PQ, "disorder": O.UPD_DIS, "ew": O.UPD_EW}


def run(ro, lx, ly, rule, n, T=0, skip=0, layout=(4, 4), p=0.6, q=0.3):
    s = (K.SchedulerDTr if ro else K.SchedulerDT)(lx, ly, threads=T, layout=layout, skip=skip)
    s.supplySeed(77)
    s.initHomogeneous()
    s.setPQ(p, q)
    s.setPQ(q, p, 1)
    m = O.Dsfmt(O.seed32(77))
    st = O.Streams(s.threads, m, S=skip or None)
    dis = None
    if rule == "disorder":
        dis = np.random.default_rng(9).integers(0, 1 << 32, s.size_words, dtype=np.uint64).astype(np.uint32)
        s.setDisorder(dis)
    {"kpz": s.mcs, "pq": s.mcsPQSyncRng, "disorder": s.mcsDisorder2SyncRng, "ew": s.mcsEW}[rule](n)
    lat = O.flat(lx, ly, O.ENC_LOCAL)
    if rule in ("kpz", "pq"):
        O.dt_mcs_threaded(lat, lx, ly, layout[0], layout[1], st, m, n, THREADS, ro, RULES[rule], p, q)
    else:
        r = O.rates([p, q, p, p], [q, p, q, q], dis)  # classes 2 and 3 were not set: class 0's rates
        O.dt_mcs_rates(lat, lx, ly, layout[0], layout[1], st, m, n, ro, RULES[rule], r)
    got = s.popSystem()
    if not np.array_equal(got, lat):
        pytest.fail(f"{np.count_nonzero(got != lat)} words differ")
    assert np.array_equal(s.streams(), st.states)
    assert s.master_draw() == m.close_open()


# 2^17 and 2^18 blocks of 4 x 4 sites
@pytest.mark.parametrize("lx,ly", [(12, 11), (12, 12)])
@pytest.mark.parametrize("ro", [False, True])
def test_draws_in_runs(ro, lx, ly):
    run(ro, lx, ly, "pq", 2, layout=(2, 2))


@pytest.mark.parametrize("ro", [False, True])
def test_draws_in_runs_16(ro):
    run(ro, 14, 14, "pq", 1)
