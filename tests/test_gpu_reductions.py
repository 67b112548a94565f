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
