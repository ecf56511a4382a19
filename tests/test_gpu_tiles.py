"""Reads to calls by tiles of 64 sites (the batched form) at the edges of its
classes: depths on both sides of every class bound and of the general path's,
piles of reads on one anchor, many short reads over one tile, N references
whose HET cap looks at the next tile's first site, and chromosomes of a few
sites.  The text is the oracle's."""
from __future__ import annotations

import random

import pytest

import oracle_lib

pytestmark = pytest.mark.gpu

L = 100
DEPTHS = [1, 15, 16, 17, 31, 32, 33, 40, 41, 63, 64, 65, 127, 128, 129, 200, 255, 256, 300]
PILES = [2, 6, 7, 8, 30, 100, 127, 128, 260]


def _reads(rng):
    """(chromosome lengths, N runs, reads as (chromosome, 0-based start, length, strand, hit))."""
    reads = []
    at = 1000
    for d in DEPTHS:  # exactly d reads over every site of a block: d layers of reads end to end
        for k in range(d):
            p = at + k % 37
            while p < at + 500:
                n = rng.choice([L, L, rng.randint(40, L)])
                reads.append(("chrA", p, n, rng.choice("+-"), 1))
                p += n
        at += 900
    for k in PILES:  # k reads on one anchor of each strand, over a little ordinary depth
        for strand in "+-":
            for _ in range(k):
                n = L if strand == "+" else rng.randint(60, L)
                reads.append(("chrA", at if strand == "+" else at + L - n, n, strand, 1))
            at += 30
        for _ in range(12):
            reads.append(("chrA", at - 120 + rng.randrange(150), L, rng.choice("+-"), rng.choice([1, 1, 2, 3])))
        at += 400
    for n_short, length in ((150, 3), (400, 10), (700, 2), (1500, 1)):  # many reads over a tile, few over a site
        for _ in range(n_short):
            reads.append(("chrA", at + rng.randrange(64), length, rng.choice("+-"), rng.choice([1, 1, 1, 2])))
        at += 400
    n_run = (at, at + 1500)
    for _ in range(900):  # unique and repeat reads over an N reference
        reads.append(("chrA", at + rng.randrange(1400), rng.randint(1, 40), rng.choice("+-"), rng.choice([1, 2, 2])))
    at += 2000
    lens = {"chrA": at + 300}
    for i, n in enumerate((2, 63, 64, 65, 128, 129, 1000)):
        c = f"chr{i}"
        lens[c] = n
        for _ in range(max(1, n // 8)):
            k = rng.randint(1, min(L, n - 1))
            reads.append((c, rng.randrange(max(1, n - k)), k, rng.choice("+-"), rng.choice([1, 1, 2])))
    return lens, n_run, reads


@pytest.mark.parametrize("tail,flags", [(0, {}), (0, {"het_novel_r": 0.6}), (1_400_000, {"rank_sum_mode": 1}),
                                        (1_400_000, {"het_novel_r": 0.6, "rank_sum_mode": 1})])
def test_tile_edges_match_oracle(built, tmp_path, tail, flags):
    """tail: uncovered sites after chrA's reads, which take its span past the
    tile count up to which every tile of at most 64 records shares a class."""
    import gsnp_amd

    rng = random.Random(97)
    lens, (n0, n1), reads = _reads(rng)
    lens["chrA"] += tail
    seqs = {c: "".join(rng.choices("ACGT", k=n)) for c, n in lens.items()}
    seqs["chrA"] = seqs["chrA"][:n0] + "N" * (n1 - n0) + seqs["chrA"][n1:]
    fa, so = tmp_path / "g.fa", tmp_path / "d.soap"
    fa.write_text("".join(f">{c}\n" + "\n".join(v[i:i + 60] for i in range(0, len(v), 60)) + "\n" for c, v in seqs.items()))
    order = {c: i for i, c in enumerate(lens)}
    reads.sort(key=lambda r: (order[r[0]], r[1]))
    lines = []
    for i, (c, p, n, strand, hit) in enumerate(reads):
        ref = seqs[c][p:p + n]
        seq = "".join(rng.choice("AG") if b == "N" else b if rng.random() >= 0.05 else rng.choice("ACGTN") for b in ref)
        q = "".join(chr(64 + rng.choice([-1, 1, 2, 40, 40, rng.randint(1, 63)])) for _ in seq)
        q = "".join(chr(65) if hit == 1 and ch == chr(63) and rng.random() < 0.5 else ch for ch in q)
        lines.append(f"r{i}\t{seq}\t{q}\t{hit}\ta\t{n}\t{strand}\t{c}\t{p + 1}\t0\n")
    so.write_text("".join(lines))
    print(f"[tiles] {len(reads)} reads, {sum(lens.values())} sites, {flags}", flush=True)
    gt, ct = tmp_path / "gpu.cns", tmp_path / "cpu.cns"
    gsnp_amd.run(fa, so, gt, batched=64, read_length=L, **flags)
    oracle_lib.run(fa, so, ct, read_length=L, **flags)
    a, b = gt.read_bytes(), ct.read_bytes()
    if a != b:
        la, lb = a.split(b"\n"), b.split(b"\n")
        bad = [i for i, (x, y) in enumerate(zip(la, lb)) if x != y]
        raise AssertionError(f"{len(la)} vs {len(lb)} rows, {len(bad)} differ, first:\n gpu    {la[bad[0]] if bad else ''}"
                             f"\n oracle {lb[bad[0]] if bad else ''}")
