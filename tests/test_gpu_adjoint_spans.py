"""The adjoint's records and gradient at the edges of its blocks of 16,384
sites, reduction chunks of 64 records and depth classes (1 to 255 records a
site): keys against the calling path's log-likelihoods and against the whole
span's, the gradient against torch autograd in 64 bits."""
from __future__ import annotations

import ctypes
import math
import random

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = 50
BLOCK, CHUNK = 16384, 64
DEPTHS = [1, 2, 7, 8, 9, 16, 17, 32, 33, 64, 65, 128, 129, 200, 400]


@pytest.fixture(scope="module")
def spans(built, tmp_path_factory):
    import gsnp_amd
    from gsnp_amd.adjoint import Adjoint

    root = tmp_path_factory.mktemp("spans")
    rng = random.Random(5)
    n = 2 * BLOCK + 700
    seq = "".join(rng.choices("ACGT", k=n))
    seq = seq[:900] + "N" * 150 + seq[1050:]
    starts = [p for p in range(0, n - L, 4)]  # about twelve reads over a site
    starts = [p for p in starts if not 700 <= p < 1200]
    for i, d in enumerate(DEPTHS):  # d - 12 more over a stretch, at either side of the blocks' bound
        for at in (2000 + 200 * i, BLOCK - 60 + 3 * i):
            starts += [at + k % 7 for k in range(max(0, d - 12))]
    starts += [1040 + 5 * k for k in range(3)]  # single records, some over the N run
    starts.sort()
    lines = []
    for i, p in enumerate(starts):
        ref = seq[p:p + L]
        s = "".join(rng.choice("AG") if b == "N" else b if rng.random() >= 0.03 else rng.choice("ACGTN") for b in ref)
        q = "".join(chr(64 + rng.choice([30, 30, 30, 40, rng.randint(1, 45)])) for _ in s)
        lines.append(f"r{i}\t{s}\t{q}\t{rng.choice([1, 1, 1, 2])}\ta\t{L}\t{rng.choice('+-')}\tc\t{p + 1}\t0\n")
    fa, so = root / "g.fa", root / "d.soap"
    fa.write_text(">c\n" + "\n".join(seq[i:i + 60] for i in range(0, n, 60)) + "\n")
    so.write_text("".join(lines))
    p0 = gsnp_amd.matrix_gen(fa, so, read_length=L)
    job = gsnp_amd.Job(fa, so, read_length=L)
    adj = Adjoint(job)
    yield job, n, p0, adj.export()
    job.close()


def test_keys_give_the_calling_likelihoods(spans):
    import gsnp_amd

    job, n, p0, (keys, off, prow) = spans
    depth = np.diff(off)
    assert {1, 255} <= set(depth.tolist()) and np.all(depth[prow == 0xFFFFFFFF] == 0)
    block = np.repeat(np.arange(n) // BLOCK, depth.astype(np.int64))
    assert np.unique(block << np.int64(16) | keys, return_counts=True)[1].max() > CHUNK
    job.call(batched=0, emit_text=False)
    lk = np.zeros((n, 10))
    out = gsnp_amd.WindowOut()
    out.lk10 = lk.ctypes.data
    gsnp_amd.check(gsnp_amd.lib().gsnp_window_results(job.ctx, n, ctypes.byref(out)))
    p = p0.reshape(256, 256, 4, 4)[:64].transpose(0, 1, 3, 2).reshape(-1, 4)  # [key][allele]
    rows = np.stack([np.log10(0.5 * p[:, a] + 0.5 * p[:, b]) for a in range(4) for b in range(a, 4)], axis=1)
    mine = np.zeros((n, 10))
    np.add.at(mine, np.repeat(np.arange(n), depth.astype(np.int64)), rows[keys])
    called = prow != 0xFFFFFFFF
    # at most 255 terms: 255 * 2^-53 relative to the sum of their sizes, all of one sign up to rounding
    assert np.allclose(mine[called], lk[called], rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("start,size", [(0, 1), (1039, 2), (0, BLOCK - 1), (0, BLOCK), (0, BLOCK + 1), (900, 150),
                                        (17, 2 * BLOCK), (2000, 3200), (0, 2 * BLOCK + 700)])
def test_span_edges_match_autograd(spans, start, size):
    import torch

    from gsnp_amd.adjoint import Adjoint, reference_loglik_torch

    job, n, p0, (keys, off, prow) = spans
    lh = math.log(job._p.het_novel_r)
    adj = Adjoint(job, 0, start, size)
    ll, grad, dh = adj.eval(p0, lh)
    k, o, r = adj.export()
    assert np.array_equal(k, keys[int(off[start]):int(off[start + size])])
    assert np.array_equal(o, off[start:start + size + 1] - off[start]) and np.array_equal(r, prow[start:start + size])
    if not k.size:
        assert np.all(grad == 0.0)
        return
    lp, mask = adj.priors(lh)
    log_p = torch.tensor(np.log(p0.reshape(256, 256, 4, 4)[:64]), dtype=torch.float64, requires_grad=True)
    log_het = torch.tensor(lh, dtype=torch.float64, requires_grad=True)
    ref = reference_loglik_torch(log_p, log_het, k, o, r, lp, mask, lh)
    ref.backward()
    assert abs(float(ref.detach()) - ll) <= 1e-11 * abs(ll) + 1e-13
    g = log_p.grad.numpy()
    assert np.allclose(grad, g, rtol=1e-9, atol=1e-12 * np.abs(g).max())
    unused = np.setdiff1d(np.arange(65536), k)
    assert np.all(grad.transpose(0, 1, 3, 2).reshape(-1, 4)[unused] == 0.0)
    assert abs(float(log_het.grad) - dh) <= 1e-9 * abs(dh) + 1e-13
    again = adj.eval(p0, lh)
    assert np.array_equal(again[1].view(np.uint64), grad.view(np.uint64))


def test_a_long_span_s_memory_is_given_back(built):
    """A span a thousandth as long as the one before it: most of the device memory that the longer one took is free
    again, and the gradient is that of the short span in a context of its own."""
    import gsnp_amd
    from gsnp_amd.adjoint import Adjoint

    hip, free, total = ctypes.CDLL("libamdhip64.so.7"), ctypes.c_size_t(), ctypes.c_size_t()

    def free_bytes():
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    pm = np.full(256 * 256 * 16, 0.02)
    pm.reshape(256, 256, 4, 4)[:, :, range(4), range(4)] = 0.94
    job = gsnp_amd.Job(synth=(4, 5, 0.25))  # 500 kb
    try:
        job.select(0)
        job.call(batched=32, emit_text=0)  # the sites' rows, which both share
        before = free_bytes()
        Adjoint(job)
        long = free_bytes()
        got = Adjoint(job, start=3000, n_sites=500).eval(pm, math.log(1e-3))
        short = free_bytes()
    finally:
        job.close()
    taken = before - long
    print(f"[adjoint] long span {taken >> 20} MiB, given back {(short - long) >> 20} MiB", flush=True)
    assert taken > 200 << 20 and short - long > taken // 2
    job = gsnp_amd.Job(synth=(4, 5, 0.25))
    try:
        ref = Adjoint(job, start=3000, n_sites=500).eval(pm, math.log(1e-3))
    finally:
        job.close()
    assert got[0] == ref[0] and got[2] == ref[2] and np.array_equal(got[1], ref[1])


def test_a_prepared_span_outlives_its_chromosome(built):
    """The context gets a chromosome without known SNPs after a span with some was prepared: the span's evaluation
    still has its own prior rows."""
    import gsnp_amd

    lib, check = gsnp_amd.lib(), gsnp_amd.check
    rng = np.random.default_rng(3)
    n, k = 3000, 900
    codes = rng.integers(0, 4, n).astype(np.uint8)
    at = np.sort(rng.choice(n, k, replace=False)).astype(np.uint32)
    codes[at] |= 8
    snps = (gsnp_amd.Snp * k)()
    for s, f in zip(snps, rng.dirichlet(np.ones(4), k)):
        s.hapmap, s.validated = 1, 1
        s.freq[:] = f
    pos = np.sort(rng.integers(0, n - L - 1, 1200)).astype(np.int32)
    m = len(pos)
    arrays = (pos, np.full(m, (L << 16) | 1, np.int32), np.full(m, ord("+"), np.uint8),
              np.frombuffer(b"ACTG", np.uint8)[codes[pos[:, None] + np.arange(L)] & 3], np.full((m, L), 64 + 30, np.uint8))
    rb = gsnp_amd.ReadBatch(m, L, *(a.ctypes.data for a in arrays))
    pm = np.full(256 * 256 * 16, 0.02)
    pm.reshape(256, 256, 4, 4)[:, :, range(4), range(4)] = 0.94
    p, ctx = gsnp_amd.params(read_length=L, refine_mode=1), ctypes.c_void_p()
    check(lib.gsnp_device_init(0))
    check(lib.gsnp_create(ctypes.byref(p), pm.ctypes.data, ctypes.byref(ctx)))
    try:
        def evaluate():
            ll, dh, g, sites, rows = ctypes.c_double(), ctypes.c_double(), np.zeros(64 * 256 * 16), np.zeros(n), ctypes.c_uint32()
            check(lib.gsnp_adjoint_eval(ctx, pm.ctypes.data, math.log(1e-3), ctypes.byref(ll), g.ctypes.data,
                                        ctypes.byref(dh), sites.ctypes.data))
            check(lib.gsnp_adjoint_info(ctx, None, None, ctypes.byref(rows)))
            return ll.value, dh.value, g, sites, rows.value

        check(lib.gsnp_set_chromosome(ctx, b"a", codes.ctypes.data, n, at.ctypes.data, ctypes.addressof(snps), k))
        check(lib.gsnp_load_reads(ctx, ctypes.byref(rb)))
        check(lib.gsnp_adjoint_prepare(ctx, 0, n))
        first = evaluate()
        assert first[4] == 8 + k
        other = np.zeros(500, np.uint8)
        check(lib.gsnp_set_chromosome(ctx, b"b", other.ctypes.data, 500, None, None, 0))
        second = evaluate()
        assert first[:2] == second[:2] and first[4] == second[4]
        assert np.array_equal(first[2], second[2]) and np.array_equal(first[3], second[3])
    finally:
        lib.gsnp_destroy(ctx)
