"""gsnp_sort_likelihood on a caller's records of every form it accepts: plain
ones (the calling launches with the sorted rows written back), and sites with
occurrence bytes other than 1, with bits above the base, or scored through an
adjusted-quality table that holds values beyond the score table (one thread
per site).  Rows and log-likelihoods are the oracle's, bit for bit."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle_lib

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 2, 8, 9, 16, 17, 32, 33, 64, 65, 128, 129, 255, 256]


@pytest.mark.parametrize("kind,n_sites", [("plain", 15), ("plain", 700), ("occurrence", 700), ("high", 700), ("all ones", 15),
                                          ("growing", 300)])
def test_sort_likelihood_forms(built, kind, n_sites):
    import gsnp_amd

    L, o = gsnp_amd.lib(), oracle_lib.orc()
    rng = np.random.default_rng(31)
    flags = {"pcr_dependency": 0.9, "global_dependency": 1.02} if kind == "growing" else {}
    p = gsnp_amd.params(read_length=100, **flags)
    pm = rng.uniform(0.01, 1.0, 256 * 256 * 16)
    ctx = ctypes.c_void_p()
    gsnp_amd.check(L.gsnp_device_init(0))
    gsnp_amd.check(L.gsnp_create(ctypes.byref(p), pm.ctypes.data, ctypes.byref(ctx)))
    try:
        most = 40 if kind == "growing" else 256
        counts = np.minimum(rng.poisson(rng.gamma(2.0, 20.0, n_sites)), most).astype(np.uint32)
        counts[:len(EDGES)] = np.minimum(EDGES, most)[:n_sites]
        recs = np.zeros((n_sites, 256), dtype=np.uint32)
        for i in range(n_sites):
            n = int(counts[i])
            cyc = rng.integers(0, 100 if i % 3 else 4, n)
            w = (rng.integers(0, 4, n) << 23) | ((64 - rng.integers(1, 31, n)) << 17) | (cyc << 9) | (rng.integers(0, 2, n) << 8)
            occ = np.ones(n, dtype=np.int64)
            if kind == "occurrence" and i % 4 == 0 and n:
                occ[rng.integers(0, n, max(1, n // 5))] = rng.choice([0, 2, 3, 200])
            if kind == "high" and i % 4 == 0 and n:
                w[rng.integers(0, n, max(1, n // 5))] |= int(rng.integers(1, 128)) << 25
            w |= occ
            if kind == "all ones" and n:
                w[: max(1, n // 3)] = 0xFFFFFFFF
            recs[i, :n] = w
        work, lk = recs.copy(), np.zeros((n_sites, 10))
        print(f"[sorted] {kind}, {n_sites} sites, {counts.sum()} records", flush=True)
        gsnp_amd.check(L.gsnp_sort_likelihood(ctx, work.ctypes.data, 256, counts.ctypes.data, n_sites, lk.ctypes.data))
        score = np.zeros(256 * 256 * 4 * 10)
        o.orc_score_table(pm.ctypes.data, score.ctypes.data)
        for i in range(n_sites):
            n = int(counts[i])
            want = np.sort(recs[i, :n])
            assert np.array_equal(work[i, :n], want), f"site {i} (n={n}) not sorted"
            ref = np.zeros(10)
            rr = np.ascontiguousarray(want)
            # the oracle counts per (strand, cycle) with the read length as stride: 256 keeps every cycle apart
            assert o.orc_likelihood_sorted(rr.ctypes.data, n, 256, p.pcr_dependency, p.global_dependency,
                                           score.ctypes.data, ref.ctypes.data) == 0
            assert np.array_equal(lk[i].view(np.uint64), ref.view(np.uint64)), f"site {i} (n={n}) likelihood differs"
    finally:
        L.gsnp_destroy(ctx)


@pytest.mark.parametrize("odd", ["every", "every other", "blocks", "last of each class"])
def test_sort_likelihood_shares_of_odd_sites(built, odd):
    """Sites whose records occur more than once among plain ones: every site (whole groups of a launch are left to
    the one-thread kernel), every other one, runs of 100, and a few in each depth class."""
    import gsnp_amd

    L, o = gsnp_amd.lib(), oracle_lib.orc()
    rng = np.random.default_rng(37)
    p = gsnp_amd.params(read_length=100)
    pm = rng.uniform(0.01, 1.0, 256 * 256 * 16)
    n_sites = 1500
    counts = np.concatenate([rng.integers(lo, hi + 1, 250) for lo, hi in
                             ((0, 8), (9, 16), (17, 32), (33, 64), (65, 128), (129, 256))]).astype(np.uint32)
    if odd != "last of each class":
        counts = rng.permutation(counts)
    i = np.arange(n_sites)
    is_odd = {"every": i >= 0, "every other": i % 2 == 1, "blocks": i // 100 % 2 == 0,
              "last of each class": i % 250 >= 247}[odd]
    shape = (n_sites, 256)
    recs = ((rng.integers(0, 4, shape) << 23) | ((64 - rng.integers(1, 31, shape)) << 17) | (rng.integers(0, 30, shape) << 9)
            | (rng.integers(0, 2, shape) << 8) | np.where(is_odd[:, None], rng.integers(1, 4, shape), 1)).astype(np.uint32)
    ctx = ctypes.c_void_p()
    gsnp_amd.check(L.gsnp_device_init(0))
    gsnp_amd.check(L.gsnp_create(ctypes.byref(p), pm.ctypes.data, ctypes.byref(ctx)))
    try:
        work, lk = recs.copy(), np.full((n_sites, 10), np.nan)
        gsnp_amd.check(L.gsnp_sort_likelihood(ctx, work.ctypes.data, 256, counts.ctypes.data, n_sites, lk.ctypes.data))
        score = np.zeros(256 * 256 * 4 * 10)
        o.orc_score_table(pm.ctypes.data, score.ctypes.data)
        for s in range(n_sites):
            n = int(counts[s])
            want, ref = np.sort(recs[s, :n]), np.zeros(10)
            assert np.array_equal(work[s, :n], want), f"site {s} (n={n}) not sorted"
            assert o.orc_likelihood_sorted(want.ctypes.data, n, 256, p.pcr_dependency, p.global_dependency,
                                           score.ctypes.data, ref.ctypes.data) == 0
            assert np.array_equal(lk[s].view(np.uint64), ref.view(np.uint64)), f"site {s} (n={n}) likelihood differs"
    finally:
        L.gsnp_destroy(ctx)
