"""Batches and servers on both sides of the rules that choose their kernels: DT
blocks with a wave each (up to 2^14 of them) or a lane each, SCABit rows shared
by 8 or, in small launches, up to 64 lanes."""
import numpy as np
import pytest

import cudakpz_amd as K

pytestmark = pytest.mark.gpu

CLS = {K.KPZ_DT: K.SchedulerDT, K.KPZ_DTR: K.SchedulerDTr, K.KPZ_SCABIT: K.SchedulerSCABit}


def alone(kind, lx, ly, p, q, seed, n):
    s = CLS[kind](lx, ly)
    s.supplySeed(seed)
    s.initHomogeneous()
    if kind != K.KPZ_SCABIT and (p, q) == (1.0, 0.0):
        s.mcs(n)
    else:
        s.setPQ(p, q)
        s.mcsPQSyncRng(n)
    return s


# 2^14 blocks in all, one replica more, and 2^16
@pytest.mark.parametrize("count", [4, 5, 16])
def test_batch_dt(count):
    reps = [(K.KPZ_DT if i & 1 else K.KPZ_DTR, 11, 11, *((1.0, 0.0) if i & 2 else (0.6, 0.3)), 50 + i)
            for i in range(count)]
    b = K.Batch(reps)
    b.initHomogeneous()
    b.mcs(2)
    for i in {0, 1, 2, 3, count - 1}:
        s = alone(*reps[i], 2)
        assert np.array_equal(b.popSystem(i), s.popSystem())
        assert np.array_equal(b.streams(i), s.streams())


# under 2^18 blocks in all, and 2^18: draws in runs
@pytest.mark.parametrize("count", [63, 64])
def test_batch_dt_runs(count):
    reps = [(K.KPZ_DT if i & 1 else K.KPZ_DTR, 11, 11, 0.6, 0.3, 50 + i) for i in range(count)]
    b = K.Batch(reps)
    b.initHomogeneous()
    b.mcs(2)
    for i in (0, 1, count - 2, count - 1):
        s = alone(*reps[i], 2)
        assert np.array_equal(b.popSystem(i), s.popSystem())
        assert np.array_equal(b.streams(i), s.streams())


# rows of 512 words: 64 lanes a row alone, 8 among many rows
@pytest.mark.parametrize("others", [0, 40])
def test_batch_row_split(others):
    reps = [(K.KPZ_SCABIT, 16, 6, 0.9, 0.1, 7)] + [(K.KPZ_SCABIT, 8, 13, 0.5, 0.5, 60 + i) for i in range(others)]
    b = K.Batch(reps)
    b.initHomogeneous()
    b.mcs(3)
    s = alone(*reps[0], 3)
    assert np.array_equal(b.popSystem(0), s.popSystem())
    assert np.array_equal(b.streams(0), s.streams())


def test_server_job_outlives_the_others():
    # the rows of the long job are shared by more lanes once the short jobs have gone
    srv = K.Server(hbm_budget=1 << 28, max_slots=64, max_tick_mcs=4)
    jobs = [(K.KPZ_SCABIT, 13, 9, 23, 0.8, 0.2, 5)]
    jobs += [(K.KPZ_SCABIT, 9, 13, 5, 0.5, 0.1, 70 + i) for i in range(30)]
    jobs += [(K.KPZ_DT, 11, 11, 9, 1.0, 0.0, 90 + i) for i in range(5)]
    ids = {srv.submit(*j, keep_lattice=True): j for j in jobs}
    while True:
        left = srv.step()
        while (r := srv.pop()) is not None:
            kind, lx, ly, n, p, q, seed = ids.pop(r.id)
            if seed in (5, 70, 99, 90, 94):
                assert np.array_equal(r.lattice, alone(kind, lx, ly, p, q, seed, n).popSystem())
        if left == 0:
            break
    assert not ids
