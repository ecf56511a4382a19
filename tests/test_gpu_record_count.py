"""The record counter of a context (gsnp_stats) after batched calls: the sum of
the called sites' unique-hit depths, for blocks of one to many waves and tiles of
every class."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = 60


@pytest.mark.parametrize("n_sites,depth,deep", [(64, 20, 0), (513, 20, 0), (5_000, 30, 0), (60_000, 30, 90),
                                                (60_000, 8, 200), (1_400_000, 12, 90)])
def test_counter_is_the_sum_of_depths(built, n_sites, depth, deep):
    """deep: depth of 400 sites in the middle."""
    import gsnp_amd

    lib, check = gsnp_amd.lib(), gsnp_amd.check
    rng = np.random.default_rng(n_sites + depth)
    k = min(L, n_sites // 2)
    pos = rng.integers(0, n_sites - k, depth * n_sites // k)
    pos = np.sort(np.append(pos, n_sites // 2 + rng.integers(0, 400, deep * 400 // k) if deep else [])).astype(np.int32)
    n = len(pos)
    arrays = (pos, np.where(rng.random(n) < 0.05, (k << 16) | 2, (k << 16) | 1).astype(np.int32),
              np.where(rng.random(n) < 0.5, ord("-"), ord("+")).astype(np.uint8),
              np.frombuffer(b"ACTG", np.uint8)[rng.integers(0, 4, (n, k))],
              rng.integers(66, 104, (n, k)).astype(np.uint8))
    rb = gsnp_amd.ReadBatch(n, k, *(a.ctypes.data for a in arrays))
    p, pm, ctx = gsnp_amd.params(read_length=L), np.full(256 * 256 * 16, 0.25), ctypes.c_void_p()
    codes, uni, got = rng.integers(0, 4, n_sites).astype(np.uint8), np.zeros(n_sites, np.int32), ctypes.c_uint64()
    check(lib.gsnp_device_init(0))
    check(lib.gsnp_create(ctypes.byref(p), pm.ctypes.data, ctypes.byref(ctx)))
    try:
        check(lib.gsnp_set_chromosome(ctx, b"c", codes.ctypes.data, n_sites, None, None, 0))
        check(lib.gsnp_load_reads(ctx, ctypes.byref(rb)))
        for _ in range(3):
            check(lib.gsnp_stats(ctx, None, 1))
            check(lib.gsnp_batched_call(ctx, 0, n_sites, 0, None))
            w = gsnp_amd.WindowOut(dep_uni=uni.ctypes.data)
            check(lib.gsnp_window_results(ctx, n_sites, ctypes.byref(w)))
            check(lib.gsnp_stats(ctx, ctypes.byref(got), 0))
            assert uni.sum() > 0 and got.value == int(uni.sum())
    finally:
        lib.gsnp_destroy(ctx)
