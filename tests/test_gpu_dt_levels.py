"""Blocks of the wave-per-block double-tiling kernel whose updates need more
levels than it applies at a time (32).  Random blocks need 12 to 25, and no skip
of the generator gives many more, so the streams here take a step of their own,
s -> a s + c with a = 1 (mod 2^(k + 2)) and c = 2^k times an odd number: the
coordinates, which are bits of s, go round a few sites and each takes many
levels.  The levels are counted on the host first."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import cudakpz_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TESTS = os.path.dirname(os.path.abspath(__file__))
AT_ONCE = 32
RULES = {"kpz": (0, O.UPD_KPZ), "pq": (1, O.UPD_PQ), "disorder": (2, O.UPD_DIS), "ew": (3, O.UPD_EW)}


def block_levels(states, a, c, draws, ro):
    """levels of every stream's next block, window by window of 64 updates"""
    s, a, c = states.copy(), np.uint64(a), np.uint64(c)
    shift = np.uint64(19 if ro else 28)
    total = np.zeros(s.size, int)
    with np.errstate(over="ignore"):
        for _ in range(4):
            done = np.zeros((s.size, 18, 18), int)
            for _ in range(64):
                xy = []
                for k in range(draws):
                    s = s * a + c
                    if k < 2:
                        fold = (s ^ (s >> np.uint64(32))) & np.uint64(0xFFFFFFFF)
                        xy.append(((fold >> shift) & np.uint64(15)).astype(int) + 1)
                t, (x, y) = np.arange(s.size), xy
                at = [done[t, x + dx, y + dy] for dx, dy in ((0, 0), (1, 0), (-1, 0), (0, 1), (0, -1))]
                done[t, x, y] = 1 + np.max(at, axis=0)
            total += done.max(axis=(1, 2))
    return total


@pytest.fixture(scope="module")
def dt_step(tmp_path_factory):
    package = os.path.dirname(K.LIB_PATH)
    out = str(tmp_path_factory.mktemp("dt_step") / "dt_step.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-I" + os.path.join(package, "csrc"), "-o", out, os.path.join(TESTS, "dt_step.cpp"), K.LIB_PATH,
                           "-Wl,-rpath," + package])
    f = C.CDLL(out).dt_step_run
    f.argtypes = [C.c_int] * 3 + [C.c_uint64] * 3 + [C.c_int] + [C.c_double] * 4 + [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p]
    return f


# all blocks need 64 or 128 levels, or some of them more than 32
@pytest.mark.parametrize("ro,k,rule", [(False, 61, "kpz"), (False, 62, "kpz"), (False, 62, "ew"), (False, 62, "pq"),
                                       (False, 59, "pq"), (False, 59, "disorder"), (True, 52, "kpz"), (True, 53, "kpz"),
                                       (True, 53, "ew"), (True, 53, "pq"), (True, 50, "pq"), (True, 50, "disorder")])
def test_more_levels_than_at_once(dt_step, ro, k, rule):
    # p = 1: every update is accepted at a minimum, so all of them take a level
    lx, ly, seed, n, p, q, q1 = 8, 7, 5, 6, 1.0, 0.5, 0.25
    m = O.Dsfmt(O.seed32(seed))
    st = O.Streams(1 << (lx + ly - 10), m, S=1)
    st.a, st.c = (1 + (5 << (k + 2))) % (1 << 64), (11 << k) % (1 << 64)
    assert block_levels(st.states, st.a, st.c, 2 if rule in ("kpz", "ew") else 3, ro).max() > AT_ONCE
    dis = None
    if rule == "disorder":
        dis = np.random.default_rng(2).integers(0, 1 << 32, 1 << (lx + ly - 4), dtype=np.uint64).astype(np.uint32) & np.uint32(0x55555555)
    got, states = np.empty(1 << (lx + ly - 4), np.uint32), np.empty(st.T, np.uint64)
    code, oracle_rule = RULES[rule]
    assert dt_step(ro, lx, ly, seed, st.a, st.c, code, p, q, 1.0, q1, None if dis is None else dis.ctypes.data, n, got.ctypes.data,
                   states.ctypes.data) == 0
    lat = O.flat(lx, ly, O.ENC_LOCAL)
    if rule in ("kpz", "pq"):
        O.dt_mcs_threaded(lat, lx, ly, 4, 4, st, m, n, 4, ro, oracle_rule, p, q)
    else:
        O.dt_mcs_rates(lat, lx, ly, 4, 4, st, m, n, ro, oracle_rule, O.rates([p, 1.0, p, p], [q, q1, q, q], dis))
    assert np.array_equal(got, lat)
    assert np.array_equal(states, st.states)
