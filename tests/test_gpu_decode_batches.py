"""-C files of more windows than one upload holds (16), back to text on the
device: the text of a batch is written while the next one is read.  The same
bytes as the host decoder's; a file that cannot be created is an error."""
from __future__ import annotations

import random

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("contigs,length", [(16, 40), (17, 40), (40, 3000), (33, 60000)])
def test_batches_give_the_same_text(built, tmp_path, contigs, length):
    """40 x 3,000 and 33 x 60,000 rows: more text in a batch than one or two 2 MB pieces."""
    import gsnp_amd

    rng = random.Random(contigs + length)
    fa, so = tmp_path / "g.fa", tmp_path / "d.soap"
    lines, ref = [], []
    for c in range(contigs):
        seq = "".join(rng.choices("ACGT", k=length))
        ref.append(f">c{c}\n{seq}\n")
        for p in sorted(rng.randrange(length - 30) for _ in range(min(length, 6000) // 8)):
            s = "".join(b if rng.random() >= 0.05 else rng.choice("ACGT") for b in seq[p:p + 30])
            q = "".join(chr(64 + rng.randint(2, 40)) for _ in s)
            lines.append(f"r\t{s}\t{q}\t{rng.choice([1, 1, 2])}\ta\t30\t{rng.choice('+-')}\tc{c}\t{p + 1}\t0\n")
    fa.write_text("".join(ref))
    so.write_text("".join(lines))
    job = gsnp_amd.Job(fa, so, read_length=30)
    job.write(tmp_path / "cols", compress=True, batched=32)
    job.close()
    gsnp_amd.decompress(tmp_path / "cols", tmp_path / "dev.cns", device=True)
    gsnp_amd.decompress(tmp_path / "cols", tmp_path / "host.cns", device=False)
    a = (tmp_path / "dev.cns").read_bytes()
    assert a.count(b"\n") == contigs * length
    assert a == (tmp_path / "host.cns").read_bytes()
    (tmp_path / "dev.cns").write_bytes(b"x" * (len(a) + 1000))  # an older, longer file
    gsnp_amd.decompress(tmp_path / "cols", tmp_path / "dev.cns", device=True)
    assert a == (tmp_path / "dev.cns").read_bytes()
    with pytest.raises(gsnp_amd.GsnpError, match="cannot create"):
        gsnp_amd.decompress(tmp_path / "cols", tmp_path / "none" / "dev.cns", device=True)


@pytest.mark.parametrize("lengths", [[40] * 16 + [3000], [40] * 16 + [60000] * 3, [30000] * 16 + [40] * 17 + [45000]])
def test_batches_of_growing_text(built, tmp_path, lengths):
    """Batches of little text, which is written in one copy, before and after ones that go through the pinned pieces."""
    import gsnp_amd

    rng = random.Random(len(lengths))
    ref, lines = [], []
    for c, n in enumerate(lengths):
        seq = "".join(rng.choices("ACGT", k=n))
        ref.append(f">c{c}\n{seq}\n")
        p = rng.randrange(n - 30)
        lines.append(f"r\t{seq[p:p + 30]}\t{'^' * 30}\t1\ta\t30\t+\tc{c}\t{p + 1}\t0\n")
    (tmp_path / "g.fa").write_text("".join(ref))
    (tmp_path / "d.soap").write_text("".join(lines))
    job = gsnp_amd.Job(tmp_path / "g.fa", tmp_path / "d.soap", read_length=30)
    job.write(tmp_path / "cols", compress=True, batched=32)
    job.close()
    gsnp_amd.decompress(tmp_path / "cols", tmp_path / "dev.cns", device=True)
    gsnp_amd.decompress(tmp_path / "cols", tmp_path / "host.cns", device=False)
    text = (tmp_path / "dev.cns").read_bytes()
    assert text.count(b"\n") == sum(lengths) and text == (tmp_path / "host.cns").read_bytes()
