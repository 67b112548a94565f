"""The kernels a double-tiling phase can take, against the oracle at the sizes
where one hands over to the other: one wave per block (up to 2^13 or 2^14 blocks
of 16 x 16 sites), one lane per block above, and the lane kernel's p/q loop that
draws in runs (from 2^18 lanes on).  Everything is compared word for word."""
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


# one block per domain set, one row or column of blocks, a workgroup not filled
# (2 blocks), fewer streams than blocks in uneven walks
@pytest.mark.parametrize("lx,ly,T", [(5, 5, 0), (5, 6, 0), (6, 5, 1), (5, 10, 3), (11, 5, 0), (9, 8, 5)])
@pytest.mark.parametrize("rule", RULES)
@pytest.mark.parametrize("ro", [False, True])
def test_wave_per_block(ro, rule, lx, ly, T):
    run(ro, lx, ly, rule, 5, T)


# the largest lattice of the wave kernel, and the smallest of the lane kernel
@pytest.mark.parametrize("lx,ly", [(12, 12), (13, 12)])
@pytest.mark.parametrize("rule", RULES)
@pytest.mark.parametrize("ro", [False, True])
def test_hand_over(ro, rule, lx, ly):
    run(ro, lx, ly, rule, 1)


def test_many_updates_of_a_site():
    """The odd skip S with A^S = -3 (mod 2^64): a stream next to the fixed point
    c/4 of s -> -3 s + c keeps its top bits for 17 draws, so the first updates
    of every block fall on one site, one level each (a block of random sites
    has 5-6 levels in its first window)."""
    mod = 1 << 64
    A, C = 2862933555777941757, 1442695040888963407
    S = 1
    for k in range(3, 64):
        if (pow(A, S, 2 << k) + 3) % (2 << k):
            S += 1 << (k - 2)
    assert pow(A, S, mod) == mod - 3 and S % 2 == 1
    _, jc = O.slcg_jump(A, C, S)
    c = A * jc % mod
    for ro in (False, True):
        s = (K.SchedulerDTr if ro else K.SchedulerDT)(7, 6, skip=S)
        s.supplySeed(5)
        s.initHomogeneous()
        m = O.Dsfmt(O.seed32(5))
        st = O.Streams(s.threads, m, S=1)
        st.a, st.c = mod - 3, c
        st.states[:] = [(c // 4 + k + (k << 62)) % mod for k in range(s.threads)]
        s.set_streams(st.states)
        s.mcs(2)
        lat = O.flat(7, 6, O.ENC_LOCAL)
        O.dt_mcs(lat, 7, 6, 4, 4, st, m, 2, ro)
        assert np.array_equal(s.popSystem(), lat)
        assert np.array_equal(s.streams(), st.states)


# 2^17 and 2^18 blocks of 4 x 4 sites
@pytest.mark.parametrize("lx,ly", [(12, 11), (12, 12)])
@pytest.mark.parametrize("ro", [False, True])
def test_draws_in_runs(ro, lx, ly):
    run(ro, lx, ly, "pq", 2, layout=(2, 2))


@pytest.mark.parametrize("ro", [False, True])
def test_draws_in_runs_16(ro):
    run(ro, 14, 14, "pq", 1)


# the largest lattice with a wave per block for the rules other than disorder
@pytest.mark.parametrize("rule", ["kpz", "pq", "ew"])
@pytest.mark.parametrize("ro", [False, True])
def test_hand_over_of_two_draws(ro, rule):
    run(ro, 12, 11, rule, 1)


# 2^19 and 2^20 blocks of 4 x 4 sites: draws behind the reads, and before them
@pytest.mark.parametrize("lx,ly", [(13, 12), (13, 13)])
def test_draws_ahead(lx, ly):
    run(False, lx, ly, "kpz", 2, layout=(2, 2))
