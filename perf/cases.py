"""Workloads of the KPZ engine as its users run them, for timing.

A case is a dict of plain values.  `listed()` are fixed ones, `draw(rng)`
gives one more of the same ranges, `prepare(case, seed)` builds what a program
holds before the call (a seeded scheduler on its lattice, a batch, a server
with its job list), `run(state)` is one pass through the public calls, and
`work(case)` what that pass cannot do without.  `exact(case, seed)` is the
answer in 64 bits for the outputs that are computed floating-point numbers
(the height moments); every other output is a lattice or an exact integer.

The four kinds of case:

* "run": one scheduler advances by `chunk` Monte-Carlo steps at a time,
  `reps` times, and samples after each chunk what `sample` says: nothing (a
  stretch between two sample times), "w2" (roughness) or "corr" (roughness
  and the autocorrelation with every tag).  The passes of one state continue
  the same run.
* "analysis": the driver's output line for a given lattice and tag
  (roughness, moments, correlations), without Monte-Carlo steps.
* "batch": an ensemble of uneven replicas, some steps and the w2 of each.
* "serve": a list of jobs handed to a server and stepped until all are done.
"""
import random

import numpy as np
import torch

import cudakpz_amd as K

_CLASSES = {"dtStatic": K.SchedulerDT, "dt": K.SchedulerDTr, "scaBit": K.SchedulerSCABit, "sca": K.SchedulerSCA}
_KINDS = {"dtStatic": K.KPZ_DT, "dt": K.KPZ_DTR, "scaBit": K.KPZ_SCABIT}


def _run(name, scheduler, lx, ly, chunk, reps=1, sample="", rule="mcs", p=1.0, q=0.0, threads=0, lbx=4, lby=4,
         rng="slcg64"):
    return {"name": name, "kind": "run", "scheduler": scheduler, "lx": lx, "ly": ly, "chunk": chunk, "reps": reps,
            "sample": sample, "rule": rule, "p": p, "q": q, "threads": threads, "lbx": lbx, "lby": lby, "rng": rng}


def listed():
    return [
        # the smallest run in use: 512^2, sums of h and h^2 after every step (a
        # program that follows one small lattice closely; launches and latency)
        _run("dt_512_every_step", "dtStatic", 9, 9, 1, 10, "w2"),
        # small checkerboard run with a deposition and an evaporation rate, sampled now and then
        _run("scabit_1024_pq", "scaBit", 10, 10, 10, 1, "w2", "pq", 0.95, 0.05),
        # disordered rates on a mid-sized lattice, half of the sites of each class
        _run("dt_2048_disorder", "dt", 11, 11, 5, 1, "w2", "disorder", 0.9, 0.1),
        # the command line's default scheduler on the size of the statistics runs
        _run("dt_4096", "dt", 12, 12, 10, 1, "w2"),
        # the TinyMT32 worker streams of the CPU schedulers, 32 of them
        _run("dt_4096_tinymt32", "dt", 12, 12, 4, 1, "", "mcs", 1.0, 0.0, 32, 4, 4, "tinymt32"),
        # checkerboard on the local encoding, its default p = .95
        _run("sca_8192", "sca", 13, 13, 8, 1, ""),
        # bit-parallel checkerboard at its default p = .5
        _run("scabit_32768", "scaBit", 15, 15, 10, 1, ""),
        # the two headline lattices: double tiling with w2, and the
        # checkerboard at p = .95, q = .05 with w2 and the autocorrelation
        _run("dt_65536", "dtStatic", 16, 16, 2, 1, "w2"),
        _run("scabit_65536_pq_corr", "scaBit", 16, 16, 2, 1, "corr", "pq", 0.95, 0.05),
        # one line of the driver's table for a large lattice with a live tag
        {"name": "analysis_16384", "kind": "analysis", "scheduler": "dt", "lx": 14, "ly": 14},
        # ensemble of uneven replicas, half double tiling and half
        # checkerboard, half KPZ and half Edwards-Wilkinson rates
        {"name": "batch_1024", "kind": "batch", "replicas": 1024, "umin": 6, "umax": 11, "chunk": 10},
        # a burst of jobs, L = 2^8..2^13
        {"name": "serve_32", "kind": "serve", "scheduler": "scaBit", "jobs": 32, "umin": 8, "umax": 13, "mcs_min": 100,
         "mcs_max": 1000},
    ]


# site updates of one pass that no drawn case exceeds (the largest listed one's)
_MOST = 2 << 32


def _log_int(rng, lo, hi):
    return int(round(2.0 ** rng.uniform(np.log2(lo), np.log2(hi))))


def draw(rng):
    pick = rng.random()
    if pick < 0.08:
        return {"kind": "analysis", "scheduler": rng.choice(["dt", "dtStatic", "scaBit"]), "lx": rng.randint(8, 15),
                "ly": rng.randint(8, 15)}
    if pick < 0.20:
        return {"kind": "batch", "replicas": _log_int(rng, 64, 1024), "umin": 6, "umax": rng.randint(8, 11),
                "chunk": rng.randint(3, 10)}
    if pick < 0.28:
        return {"kind": "serve", "scheduler": rng.choice(["scaBit", "scaBit", "dt"]), "jobs": rng.randint(8, 32), "umin": 8,
                "umax": rng.randint(9, 12), "mcs_min": 100, "mcs_max": rng.randint(200, 600)}
    scheduler = rng.choice(["dtStatic", "dtStatic", "dt", "dt", "scaBit", "scaBit", "sca"])
    # log2 of the sides, square or up to 16 times as wide as high or the other way round
    s = rng.uniform(18.0, 32.0)
    d = rng.choice([0, 0, 1, 2, 3, 4])
    lx = min(16, max(7, int(round((s + rng.choice([-d, d])) / 2))))
    ly = min(16, max(6, int(round(s)) - lx))
    rule = rng.choice(["mcs", "mcs", "pq", "pq", "disorder"])
    p = round(rng.uniform(0.5, 1.0), 3)
    q = rng.choice([0.0, round(1.0 - p, 3), round(rng.uniform(0.0, 0.5), 3)])
    lbx, lby = (4, 4) if rng.random() < 0.8 else rng.choice([(3, 4), (4, 3), (3, 3), (2, 2)])
    # worker streams: one per block / row / column, or the thread count of some CPU run
    most = {"scaBit": 1 << ly, "sca": 1 << (lx - 2)}.get(scheduler, 1 << 16)
    threads = 0 if rng.random() < 0.65 else min(most, rng.choice([7, 32, 96, 1000]))
    stream = "slcg64"
    if scheduler != "dtStatic" and rule != "disorder" and lx + ly <= 26 and rng.random() < 0.2:
        stream, threads = "tinymt32", min(most, rng.choice([32, 96, 1000]))
        lbx = lby = 4
    reps = rng.choice([1, 1, 1, 4])
    chunk = min(_log_int(rng, 1, 40), max(1, (_MOST >> (lx + ly)) // reps))
    if chunk * reps << (lx + ly) > _MOST:
        reps = 1
    c = _run("", scheduler, lx, ly, chunk, reps, rng.choice(["", "w2", "w2", "corr"]), rule, p, q, threads, lbx, lby, stream)
    del c["name"]
    return c


class _DeviceLattice:
    """The engine's lattice as a device array (no copy); keeps its owner."""

    def __init__(self, s):
        self.owner = s
        self.__cuda_array_interface__ = {"shape": (s.size_words,), "typestr": "<i4", "data": (s.device_lattice, False),
                                         "version": 2, "strides": None}


def _lattice(s):
    return torch.as_tensor(_DeviceLattice(s), device="cuda")


def _prepare_run(case, seed):
    r = np.random.default_rng(seed)
    s = _CLASSES[case["scheduler"]](case["lx"], case["ly"], threads=case["threads"], layout=(case["lbx"], case["lby"]),
                                    rng=K.RNG_TINYMT32 if case["rng"] == "tinymt32" else K.RNG_SLCG64)
    if case["rng"] == "tinymt32":
        s.setTinyMTParams(*(r.integers(0, 1 << 32, s.threads, dtype=np.uint64).astype(np.uint32) for _ in range(3)))
    s.supplySeed(int(r.integers(1, 1 << 31)))
    s.initHomogeneous()
    if case["rule"] == "pq":
        s.setPQ(case["p"], case["q"])
    elif case["rule"] == "disorder":
        # class 0 with (p, q), class 1 (half of the sites) with the rates exchanged
        s.setPQ(case["p"], case["q"])
        s.setPQ(case["q"], case["p"], 1)
        m = r.integers(0, 1 << 32, s.size_words, dtype=np.uint64).astype(np.uint32) & np.uint32(0x55555555)
        s.setDisorder(m)
    advance = {"mcs": s.mcs, "pq": s.mcsPQSyncRng, "disorder": s.mcsDisorder2SyncRng}[case["rule"]]
    # a surface that has left the flat start behind
    advance(4 if case["lx"] + case["ly"] <= 28 else 2)
    if case["sample"] == "corr":
        s.correlateTag()
        advance(1)
    s.sync()
    return {"s": s, "advance": advance, "case": case, "lattice": _lattice(s)}


def _run_run(st):
    s, c = st["s"], st["case"]
    sums = []
    for _ in range(c["reps"]):
        st["advance"](c["chunk"])
        if c["sample"]:
            w = s.roughness()
            sums += [w.sum_h, w.sum_h2]
        if c["sample"] == "corr":
            for t, k in s.correlateAll():
                sums += [t, k.sum_h, k.sum_hs, k.sum_h2, k.sum_hhs, k.tcs]
    return {"lattice": st["lattice"], "sums": sums}


# ---- analysis: a rough surface h(x, y) = F(x) + G(y) with exactly known sums
def _walk(r, n):
    """n slopes (0 / 1), each 64 of them with as many ups as downs: a walk that
    wanders by several units and closes around the lattice"""
    w = min(64, n)
    a = np.tile(np.arange(w) < w // 2, (n // w, 1)).astype(np.uint8)
    return r.permuted(a, axis=1).reshape(-1)


def _slopes(case, seed):
    r = np.random.default_rng(seed)
    return [(_walk(r, 1 << case["lx"]), _walk(r, 1 << case["ly"])) for _ in range(2)]


def _words(bits):
    """32 slopes to a word, the first in bit 0"""
    return np.packbits(bits.reshape(-1, 32), axis=1, bitorder="little").view("<u4").reshape(-1)


def _pack(f, g, scheduler, lx, ly):
    """The lattice with x slopes f(x) and y slopes g(y)"""
    if scheduler == "scaBit":
        half = [_words(f[0::2]), _words(f[1::2])]  # the two sublattices of an even row
        q = np.empty((4, 1 << ly, 1 << (lx - 6)), np.uint32)  # (sublattice 0, 1) x (x, y slopes)
        for sub in (0, 1):
            q[2 * sub, 0::2] = half[sub]
            q[2 * sub, 1::2] = half[1 - sub]
            q[2 * sub + 1] = (g.astype(np.uint32) * np.uint32(0xFFFFFFFF))[:, None]
        return q.reshape(-1)
    # 4 x 4 sites to a word, bit 2 (x & 3) + 8 (y & 3), the y slope one above
    fx = f.reshape(-1, 4).astype(np.uint32)
    gy = g.reshape(-1, 4).astype(np.uint32)
    col = sum(fx[:, i] << np.uint32(2 * i) for i in range(4)) * np.uint32(0x01010101)
    row = sum((gy[:, j] * np.uint32(0xAA)) << np.uint32(8 * j) for j in range(4))
    return (row[:, None] | col[None, :]).reshape(-1)


def _prepare_analysis(case, seed):
    s = _CLASSES[case["scheduler"]](case["lx"], case["ly"])
    s.supplySeed(1 + seed % (1 << 31))
    (f0, g0), (f1, g1) = _slopes(case, seed)
    s.pushSystem(_pack(f0, g0, case["scheduler"], case["lx"], case["ly"]))
    s.correlateTag()
    s.pushSystem(_pack(f1, g1, case["scheduler"], case["lx"], case["ly"]))
    return {"s": s, "case": case, "lattice": _lattice(s)}


def _run_analysis(st):
    s = st["s"]
    w = s.roughness()
    m = s.moments()
    corr = [[t, k.sum_h, k.sum_hs, k.sum_h2, k.sum_hhs, k.tcs] for t, k in s.correlateAll()]
    return {"lattice": st["lattice"], "w2": [w.sum_h, w.sum_h2], "moments": m, "corr": corr}


def _exact_analysis(case, seed):
    f, g = _slopes(case, seed)[1]
    up = 2 * f.astype(np.int64) - 1
    # heights: the row starts at the sum of the y slopes so far; the x slopes
    # of x >= 1 add up from there, and x = 0 closes the row (slopes sum to 0)
    F = np.concatenate([[0], np.cumsum(up[1:])])
    G = np.cumsum(2 * g.astype(np.int64) - 1)
    pf = [int((F ** k).sum()) for k in range(8)]
    pg = [int((G ** k).sum()) for k in range(8)]
    from fractions import Fraction
    from math import comb
    n = 1 << (case["lx"] + case["ly"])
    m = [float(Fraction(sum(comb(k, j) * pf[j] * pg[k - j] for j in range(k + 1)), n)) for k in range(1, 8)]
    return {"lattice": None, "w2": None, "moments": m, "corr": None}


# ---- batch
def _replicas(case, seed):
    r = random.Random(seed)
    # the mix of sizes is the case's, the seeds are the inputs
    sizes = random.Random(4096 + case["replicas"])
    reps = []
    for i in range(case["replicas"]):
        u = sizes.randint(case["umin"], case["umax"])
        kind = K.KPZ_DT if i % 2 == 0 else K.KPZ_SCABIT
        p, q = (1.0, 0.0) if (i // 2) % 2 == 0 else (0.5, 0.5)
        reps.append((kind, u, u, p, q, r.randrange(1, 1 << 31)))
    return reps


def _prepare_batch(case, seed):
    b = K.Batch(_replicas(case, seed))
    b.initHomogeneous()
    b.mcs(case["chunk"])
    b.sync()
    return {"b": b, "case": case}


def _run_batch(st):
    b = st["b"]
    b.mcs(st["case"]["chunk"])
    sums = np.array([(w.sum_h, w.sum_h2) for w in b.roughness()], dtype=np.int64)
    # one replica of each kind and rate is looked at in full
    return {"sums": sums, "lattices": [b.popSystem(i).view(np.int32) for i in range(4)]}


# ---- serving
def _jobs(case, seed):
    r = np.random.default_rng(seed)
    shape = np.random.default_rng(1000 * case["jobs"] + case["umax"])  # sizes and lengths are the case's
    out = []
    for _ in range(case["jobs"]):
        u = int(shape.integers(case["umin"], case["umax"] + 1))
        mcs = int(round(np.exp(shape.uniform(np.log(case["mcs_min"]), np.log(case["mcs_max"])))))
        p = float(r.uniform(0.5, 1.0))
        out.append((_KINDS[case["scheduler"]], u, u, mcs, p, 1.0 - p, int(r.integers(1, 1 << 31))))
    return out


def _prepare_serve(case, seed):
    return {"srv": K.Server(hbm_budget=1 << 30, max_slots=64, max_tick_mcs=16), "jobs": _jobs(case, seed)}


def _run_serve(st):
    srv = st["srv"]
    ids = {}
    for i, j in enumerate(st["jobs"]):
        ids[srv.submit(*j)] = i
    series = [None] * len(ids)
    while True:
        left = srv.step()
        while True:
            r = srv.pop()
            if r is None:
                break
            series[ids[r.id]] = [v for m, w in r.series for v in (m, w.sum_h, w.sum_h2)]
        if left == 0:
            return {"series": np.array([v for s in series for v in s], dtype=np.int64)}


_PREPARE = {"run": _prepare_run, "analysis": _prepare_analysis, "batch": _prepare_batch, "serve": _prepare_serve}
_RUN = {"run": _run_run, "analysis": _run_analysis, "batch": _run_batch, "serve": _run_serve}


def prepare(case, seed):
    st = _PREPARE[case["kind"]](case, seed)
    st["kind"] = case["kind"]
    return st


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    return _exact_analysis(case, seed) if case["kind"] == "analysis" else None


def work(case):
    """Bytes: 2 bits per site, read and written once per pass (read only in
    the analysis, with its tag).  Operations: integer ones, counted coarsely
    per site update: a double-tiling update draws two coordinates and tests
    and flips one site (30), a checkerboard site draws and compares one number
    (10) or, bit-parallel, shares its word's work with 63 others (1/2)."""
    if case["kind"] == "analysis":
        n = 1 << (case["lx"] + case["ly"])
        return {"bytes": n / 2, "flops": 20 * n}
    if case["kind"] == "batch":
        n = sum(1 << (r[1] + r[2]) for r in _replicas(case, 0))
        return {"bytes": n / 2, "flops": 20 * n * case["chunk"]}
    if case["kind"] == "serve":
        jobs = _jobs(case, 0)
        ops = 10 if case["scheduler"] == "scaBit" else 30
        return {"bytes": sum(1 << (j[1] + j[2]) for j in jobs) / 2, "flops": ops * sum(j[3] << (j[1] + j[2]) for j in jobs)}
    n = 1 << (case["lx"] + case["ly"])
    if case["scheduler"] in ("dt", "dtStatic"):
        ops = 30
    else:
        ops = 0.5 if case["scheduler"] == "scaBit" and case["rule"] == "mcs" else 10
    return {"bytes": n / 2, "flops": ops * n * case["chunk"] * case["reps"]}
