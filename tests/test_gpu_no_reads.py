"""Batched calls of a chromosome that has no reads: in a context that never
held any, after another chromosome's reads, after a batch that was rejected,
and with no chromosome at all.  The rows are the oracle's."""
from __future__ import annotations

import ctypes
import random

import numpy as np
import pytest

import oracle_lib

pytestmark = pytest.mark.gpu

L = 50


def _batch(pos):
    """Reads of L bases A, quality 30, on '+' and unique, at the given starts."""
    n = len(pos)
    keep = (np.asarray(pos, np.int32), np.full(n, (L << 16) | 1, np.int32), np.full(n, ord("+"), np.uint8),
            np.full(n * L, ord("A"), np.uint8), np.full(n * L, 64 + 30, np.uint8))
    import gsnp_amd

    return gsnp_amd.ReadBatch(n, L, *(a.ctypes.data for a in keep)), keep


@pytest.mark.parametrize("before", ["nothing", "empty_batch", "other_reads", "rejected_batch"])
def test_chromosome_without_reads_matches_oracle(built, tmp_path, before):
    import gsnp_amd

    rng = random.Random(31)
    seqs = {"chrA": "".join(rng.choices("ACGT", k=3000)), "chrB": "".join(rng.choices("ACGTN", k=gsnp_amd.WIN + 5000))}
    fa, so, out = tmp_path / "g.fa", tmp_path / "d.soap", tmp_path / "cpu.cns"
    fa.write_text("".join(f">{c}\n{s}\n" for c, s in seqs.items()))
    # the readers drop a read over the last site, so chrB is written and uncovered
    so.write_text("".join(f"r\t{'A' * L}\t{'^' * L}\t1\ta\t{L}\t+\t{c}\t{p}\t0\n"
                          for c, p in (("chrA", 101), ("chrB", len(seqs["chrB"]) - L + 1))))
    oracle_lib.run(fa, so, out, read_length=L)
    want = b"".join(r for r in out.read_bytes().splitlines(keepends=True) if r.startswith(b"chrB\t"))

    lib, check = gsnp_amd.lib(), gsnp_amd.check
    p, pm, ctx = gsnp_amd.params(read_length=L), np.full(256 * 256 * 16, 0.25), ctypes.c_void_p()
    check(lib.gsnp_device_init(0))
    check(lib.gsnp_create(ctypes.byref(p), pm.ctypes.data, ctypes.byref(ctx)))
    try:
        codes = {c: np.frombuffer(s.encode(), np.uint8) >> 1 & 7 for c, s in seqs.items()}

        def chromosome(c):
            check(lib.gsnp_set_chromosome(ctx, c.encode(), codes[c].ctypes.data, len(codes[c]), None, None, 0))

        if before == "nothing":  # no chromosome either
            check(lib.gsnp_batched_call(ctx, 0, 0, 0, None))
        if before in ("other_reads", "rejected_batch"):
            chromosome("chrA")
            rb, _keep = _batch(range(0, 2900, 10))
            check(lib.gsnp_load_reads(ctx, ctypes.byref(rb)))
            check(lib.gsnp_batched_call(ctx, 0, 3000, 0, None))
        chromosome("chrB")
        if before == "rejected_batch":
            rb, _keep = _batch([200, 100])
            assert lib.gsnp_load_reads(ctx, ctypes.byref(rb)) == 3  # unsorted
        if before == "empty_batch":
            rb, _keep = _batch([])
            check(lib.gsnp_load_reads(ctx, ctypes.byref(rb)))
        nb = ctypes.c_uint64()
        check(lib.gsnp_batched_call(ctx, 0, len(codes["chrB"]), 1, ctypes.byref(nb)))
        buf = ctypes.create_string_buffer(max(1, nb.value))
        check(lib.gsnp_fetch_text(ctx, buf, nb.value, ctypes.byref(nb)))
        got = buf.raw[:nb.value]
        assert got == want, f"{len(got)} vs {len(want)} bytes"
    finally:
        lib.gsnp_destroy(ctx)
