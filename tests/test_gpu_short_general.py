"""Short spans through the launches per depth class (an adjusted-quality table
too large for the tiles): classes that no site can reach are not launched, so
depths on both sides of each class bound at one place.  The text is the
oracle's."""
from __future__ import annotations

import random

import pytest

import oracle_lib
from test_gpu_parity import _job_text

pytestmark = pytest.mark.gpu

L, N = 100, 5000


@pytest.mark.parametrize("depth", [1, 8, 9, 16, 17, 32, 33, 64, 65, 128, 129, 255, 300])
def test_depth_bounds_match_oracle(built, tmp_path, depth):
    """depth reads over site 2047 (0-based), whose reads start in the block of 1,024 sites before and in its own."""
    import gsnp_amd

    rng = random.Random(depth)
    ref = "".join(rng.choices("ACGT", k=N))
    starts = sorted([2047 - rng.randrange(L) for _ in range(depth)] + [100, 4000])
    so = []
    for i, p in enumerate(starts):
        seq = "".join(b if rng.random() >= 0.03 else rng.choice("ACGTN") for b in ref[p:p + L])
        q = "".join(chr(64 + rng.randint(2, 40)) for _ in seq)
        so.append(f"r{i}\t{seq}\t{q}\t1\ta\t{L}\t{rng.choice('+-')}\tchr1\t{p + 1}\t0\n")
    (tmp_path / "g.fa").write_text(f">chr1\n{ref}\n")
    (tmp_path / "d.soap").write_text("".join(so))
    flags = {"read_length": L, "global_dependency": 0.95}
    oracle_lib.run(tmp_path / "g.fa", tmp_path / "d.soap", tmp_path / "cpu.cns", **flags)
    job = gsnp_amd.Job(tmp_path / "g.fa", tmp_path / "d.soap", **flags)
    try:
        job.select(0)
        job.profile(enable=True)
        job.call(batched=64)
        assert job.profile(enable=False)["site_build"][1] == 1
        assert _job_text(job) == (tmp_path / "cpu.cns").read_bytes()
    finally:
        job.close()
