"""Batched calls of spans on both sides of the choice between the tile kernels
and the launches per depth class: which of the two a span takes is read off the
stage counts, and either way the text is the oracle's."""
from __future__ import annotations

import random

import pytest

import oracle_lib
from test_gpu_parity import _job_text

pytestmark = pytest.mark.gpu

N = 12_000


@pytest.mark.parametrize("read_len,depth,deep,tiles", [
    (100, 30, None, True), (100, 60, None, True), (100, 110, None, False), (100, 220, None, False),
    (36, 40, None, True), (36, 60, None, False), (36, 100, None, False), (200, 90, None, True), (200, 150, None, False),
    (100, 20, (130, 1000), True), (100, 20, (130, 6000), False), (100, 3, (700, 300), True), (36, 8, (110, 600), True)])
@pytest.mark.parametrize("rank", [0, 1])
def test_route_and_text(built, tmp_path, read_len, depth, deep, tiles, rank):
    """deep: (depth, sites) of a part of the chromosome.  600 sites of 36 bp reads at 110x are tiles of some 300
    unique-hit reads in a span that stays with the tiles."""
    import gsnp_amd

    rng = random.Random(41)
    ref = "".join(rng.choices("ACGT", k=N))
    starts = [rng.randrange(N - read_len) for _ in range(depth * N // read_len)]
    if deep:
        starts += [5000 + rng.randrange(deep[1]) for _ in range(deep[0] * deep[1] // read_len)]
    lines = []
    for i, p in enumerate(sorted(starts)):
        n = rng.choice([read_len, read_len, rng.randint(read_len // 2, read_len)])
        seq = "".join(b if rng.random() >= 0.04 else rng.choice("ACGTN") for b in ref[p:p + n])
        q = "".join(chr(64 + rng.randint(2, 40)) for _ in seq)
        lines.append(f"r{i}\t{seq}\t{q}\t{rng.choice([1] * 12 + [2])}\ta\t{n}\t{rng.choice('+-')}\tchr1\t{p + 1}\t0\n")
    fa, so, out = tmp_path / "g.fa", tmp_path / "d.soap", tmp_path / "cpu.cns"
    fa.write_text(f">chr1\n{ref}\n")
    so.write_text("".join(lines))
    flags = {"read_length": read_len, "rank_sum_mode": rank}
    oracle_lib.run(fa, so, out, **flags)
    job = gsnp_amd.Job(fa, so, **flags)
    try:
        job.select(0)
        job.profile(enable=True)
        job.call(batched=64)
        built_rows = job.profile(enable=False)["site_build"][1]
        text = _job_text(job)
    finally:
        job.close()
    assert text == out.read_bytes()
    assert (built_rows == 0) == tiles
