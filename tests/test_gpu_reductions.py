"""Roughness and correlator on random lattices against the oracle's row-wise
sums, at the sizes where the kernels change: the words per lane of the row
statistics (narrow rows), one pass or two over the rows (1024 rows), and the
per-site or the table correlator (2^25 sites)."""
import os

import numpy as np
import pytest

import cudakpz_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu

THREADS = max(1, min(16, os.cpu_count() or 1))
CASES = [(K.SchedulerDT, O.ENC_LOCAL), (K.SchedulerSCABit, O.ENC_CBBIT)]


def random_lattice(s, seed):
    return np.random.default_rng(seed).integers(0, 1 << 32, s.size_words, dtype=np.uint64).astype(np.uint32)


@pytest.mark.parametrize("lx,ly", [(6, 5), (7, 6), (8, 9), (9, 10), (10, 11), (11, 5), (12, 7), (13, 10), (14, 6), (7, 13)])
@pytest.mark.parametrize("cls,enc", CASES)
def test_roughness(cls, enc, lx, ly):
    s = cls(lx, ly)
    lat = random_lattice(s, lx * 31 + ly)
    s.pushSystem(lat)
    r = s.roughness()
    assert (r.sum_h, r.sum_h2) == O.roughness_rows(lat, enc, lx, ly, THREADS)


@pytest.mark.parametrize("lx,ly", [(6, 7), (9, 10), (9, 11), (12, 12), (13, 12), (18, 7), (7, 18), (14, 11)])
@pytest.mark.parametrize("cls,enc", CASES)
def test_correlate(cls, enc, lx, ly):
    s = cls(lx, ly)
    snap, lat = random_lattice(s, 1), random_lattice(s, 2)
    s.pushSystem(snap)
    s.correlateTag()
    s.pushSystem(lat)
    c = s.correlate()
    assert (c.sum_h, c.sum_hs, c.sum_h2, c.sum_hhs, c.tcs) == O.correlate_rows(lat, snap, enc, lx, ly, THREADS)


# rows of 64 sites (the first with the 8-site walks) to several rounds per row,
# fewer and more rows than one group of partial sums; heights up to thousands
# from slopes of one sign in a row
@pytest.mark.parametrize("lx,ly", [(6, 2), (6, 7), (7, 5), (9, 6), (10, 5), (12, 6), (13, 3), (15, 4), (5, 6)])
@pytest.mark.parametrize("cls,enc", [(K.SchedulerSCA, O.ENC_LOCAL), (K.SchedulerSCABit, O.ENC_CBBIT)])
@pytest.mark.parametrize("steep", [False, True])
def test_moments(cls, enc, lx, ly, steep):
    if (cls is K.SchedulerSCA and ly < 3) or (cls is K.SchedulerSCABit and lx < 6):
        pytest.skip("size below the scheduler's smallest")
    s = cls(lx, ly)
    lat = random_lattice(s, lx + 40 * ly)
    if steep:
        lat |= random_lattice(s, 3) | random_lattice(s, 4)
    s.pushSystem(lat)
    got = s.moments()
    h = O.heights(lat, enc, lx, ly).astype(np.int64).ravel()
    values, counts = np.unique(h, return_counts=True)
    for k in range(1, 8):
        exact = sum(int(v) ** k * int(c) for v, c in zip(values, counts))
        size = sum(abs(int(v)) ** k * int(c) for v, c in zip(values, counts))
        # every power and sum below 2^53 is exact; beyond, some ten roundings per
        # site and level of the sums, each half an ulp of the absolute sum
        assert abs(got[k - 1] * h.size - exact) <= 2.0 ** -52 * 16 * size
