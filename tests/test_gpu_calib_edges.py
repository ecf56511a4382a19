"""Calibration counts at the edges of the counting kernel's four-base lanes and
16-cycle slices: reads of every length up to the limit on both strands, at the
first and the last site, over an N run, next to repeat hits; against a plain
count of the text (which leaves out reads that cover the last site, as the
readers do)."""
from __future__ import annotations

import random

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CODE = {"A": 0, "C": 1, "T": 2, "G": 3}


@pytest.mark.parametrize("L,n_reads", [(1, 40), (2, 40), (3, 60), (4, 60), (5, 200), (15, 300), (16, 1023), (17, 1025),
                                       (100, 9000), (255, 700), (256, 1500)])
def test_counts_are_the_text_s(built, tmp_path, L, n_reads):
    import gsnp_amd

    rng = random.Random(100 * L + n_reads)
    n = 2 * L + 900
    seq = "".join(rng.choices("ACGT", k=n))
    seq = seq[:300] + "N" * 20 + seq[320:]
    reads = []
    for k in range(1, L + 1):  # every length at either end of the reference
        for strand in "+-":
            reads += [(0, k, strand, 1), (n - k, k, strand, 1)]
    for _ in range(n_reads):
        k = rng.choice([L, L, rng.randint(1, L)])
        reads.append((rng.randrange(n - k + 1), k, rng.choice("+-"), rng.choice([1, 1, 1, 2])))
    reads.sort(key=lambda r: r[0])
    want = np.zeros((64, 256, 4, 4), np.uint64)  # quality, cycle, reference, observed
    lines = []
    for i, (p, k, strand, hit) in enumerate(reads):
        s = "".join(rng.choice("ACGTN") if rng.random() < 0.1 or b == "N" else b for b in seq[p:p + k])
        q = [rng.choice([1, 2, 40, 40, rng.randint(1, 60)]) for _ in s]
        lines.append(f"r{i}\t{s}\t{''.join(chr(64 + x) for x in q)}\t{hit}\ta\t{k}\t{strand}\tc\t{p + 1}\t0\n")
        for j in range(k):
            if hit == 1 and p + k < n and s[j] != "N" and seq[p + j] != "N":  # a read over the last site is not taken
                want[q[j], k - 1 - j if strand == "-" else j, CODE[seq[p + j]], CODE[s[j]]] += 1
    fa, so = tmp_path / "g.fa", tmp_path / "d.soap"
    fa.write_text(f">c\n{seq}\n")
    so.write_text("".join(lines))
    print(f"[calib] {len(reads)} reads of at most {L}", flush=True)
    job = gsnp_amd.Job(fa, so, read_length=L)
    job.select(0)
    got = np.full(64 << 12, 7, np.uint64)  # the counts are added to what is there
    gsnp_amd.check(gsnp_amd.lib().gsnp_calib_count(job.ctx, got.ctypes.data))
    job.close()
    assert int(want.sum()) > 0 and np.array_equal(got.reshape(want.shape) - np.uint64(7), want)
