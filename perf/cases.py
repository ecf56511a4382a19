"""Cases that stand for the calling framework in use, each one pass through its public entry points.

Kinds:

* ``rows``     -- spans called, their .cns rows formatted on the device and fetched into the caller's pinned buffer;
* ``calls``    -- spans called, the per-site calls fetched into the caller's arrays (no text);
* ``columns``  -- the -C column chunks of every window handed to the caller's callback, which keeps their bytes;
* ``windows``  -- the reference's window interface: init, update, likelihood, posterior, results, recycle per window;
* ``sorted``   -- the segmented sort and likelihood on the caller's own device records;
* ``adjoint``  -- one evaluation of the calling likelihood and its gradient on a prepared span;
* ``span``     -- a new adjoint span prepared and evaluated once;
* ``counts``   -- the pass-1 calibration counts of the loaded reads;
* ``decode``   -- -C files on disk back to .cns text, rebuilt on the device.

Workloads are the seeded generator's (``config`` 1 to 5, genome length times ``scale``, as the benchmark takes them),
or reads and records drawn here where a plain 64-bit statement of the outputs needs them.
"""
from __future__ import annotations

import ctypes
import math
import tempfile
from pathlib import Path

import numpy as np
import torch

import gsnp_amd
from gsnp_amd.adjoint import Adjoint

# nominal sites, mean depth and read length of each generator configuration at scale 1
SITES = {1: 1e5, 2: 1e7, 3: 1.52e8, 4: 2e6, 5: 2.48e8}
DEPTH = {1: 20, 2: 30, 3: 30, 4: 30, 5: 30}
READ = {1: 100, 2: 100, 3: 100, 4: 100, 5: 150}
GENOTYPES = [(a, b) for a in range(4) for b in range(a, 4)]  # AA AC AT AG CC CT CG TT TG GG (A0 C1 T2 G3)
ROW_BYTES = 60  # of one .cns row, about
# a program's buffers, allocated before it knows the sizes of its results and zero beyond them: sites of a sample
# (the contigs of config 3 differ with the seed), bytes of a row, bytes of -C chunks a site, -C windows
ROW_ROOM, CHUNK_ROOM, WINDOW_ROOM = 76, 10, 512


def listed():
    return [
        # a small region or a plasmid: one short span, bound by launches and latency
        {"name": "rows_100k", "kind": "rows", "config": 1, "scale": 1.0, "per": 32},
        # a bacterial-size chromosome with known SNPs in refine mode, rows to the caller's file buffer
        {"name": "rows_4M_refine", "kind": "rows", "config": 2, "scale": 0.41, "per": 32, "refine_mode": 1},
        # a small sample of one miscalibrated lane, called as haploid with transitions favoured
        {"name": "calls_1M_monoploid", "kind": "calls", "config": 4, "scale": 0.53, "per": 8, "is_monoploid": 1,
         "transition_dominant": 1},
        # a whole sample of many contigs of uneven depth, with repeats and gaps: the benchmark's workload, calls kept in memory
        {"name": "calls_24_contigs", "kind": "calls", "config": 3, "scale": 0.12, "per": 32},
        # one long chromosome of 150 bp pairs with the rank-sum test
        {"name": "calls_25M_150bp", "kind": "calls", "config": 5, "scale": 0.1, "per": 32, "rank_sum_mode": 1},
        # the compressed output of a sample of many contigs
        {"name": "columns_24_contigs", "kind": "columns", "config": 3, "scale": 0.06, "per": 32},
        # a caller of the reference's own window loop, ragged reads, a partial last window
        {"name": "windows_700k", "kind": "windows", "sites": 700_001, "depth": 30, "read": 100},
        # a serving loop that holds its own records and may not allocate
        {"name": "sorted_200k", "kind": "sorted", "sites": 200_003, "depth": 30},
        # one step of a refit of the calibration table
        {"name": "adjoint_2M", "kind": "adjoint", "config": 4, "scale": 1.0, "site_terms": False},
        # a new span of the refit, prepared and evaluated once
        {"name": "span_200k", "kind": "span", "config": 4, "scale": 0.1},
        # pass 1 of a run without a calibration file
        {"name": "counts_15M_150bp", "kind": "counts", "config": 5, "scale": 0.06},
        # compressed files back to text
        {"name": "decode_2M", "kind": "decode", "config": 2, "scale": 0.2, "refine_mode": 1},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["rows", "calls", "calls", "calls", "columns", "windows", "sorted", "adjoint", "span", "counts", "decode"])
    if kind == "windows":
        return {"kind": kind, "sites": int(_log(rng, 5_000, 900_000)), "depth": rng.choice([8, 20, 30, 45]),
                "read": rng.choice([50, 75, 100, 150])}
    if kind == "sorted":
        return {"kind": kind, "sites": int(_log(rng, 1_000, 262_144)), "depth": rng.choice([5, 15, 30, 60])}
    top = {"rows": 4.5e6, "calls": 2e7, "columns": 9e6, "adjoint": 2e6, "span": 1e6, "counts": 1.5e7, "decode": 2e6}[kind]
    config = 4 if kind in ("adjoint", "span") else rng.choice([1, 2, 3, 4, 5])
    sites = _log(rng, 4.8e5 if config == 3 else 4e4, top)  # 24 contigs: not all at the generator's shortest length
    c = {"kind": kind, "config": config, "scale": round(sites / SITES[config], 9)}
    if kind in ("rows", "calls", "columns"):
        c["per"] = rng.choice([4, 8, 32])
    if kind in ("rows", "calls", "columns", "decode"):
        for flag, share in (("refine_mode", 0.4), ("rank_sum_mode", 0.4), ("transition_dominant", 0.2), ("is_monoploid", 0.15)):
            if rng.random() < share:
                c[flag] = 1
    if kind == "adjoint":
        c["site_terms"] = rng.random() < 0.5
    return c


# ---- what a program has in hand ---------------------------------------------


class _State:
    """The case with its job or context, inputs and buffers; closes what it opened."""

    def __init__(self, case):
        self.case = case
        self.kind = case["kind"]
        self.job = self.ctx = self.tmp = None

    def __del__(self):
        if self.job is not None:
            self.job.close()
        elif self.ctx is not None:
            gsnp_amd.lib().gsnp_destroy(self.ctx)
        if self.tmp is not None:
            self.tmp.cleanup()


def _pinned(n, dtype=torch.uint8):
    return torch.zeros(max(1, int(n)), dtype=dtype, pin_memory=True)


def _room(case):
    """Sites that the buffers of a generated sample are made for."""
    sites = SITES[case["config"]] * case["scale"]
    return int(2 * sites) + 24_000 if case["config"] == 3 else max(1000, math.floor(sites)) + 1


def _p_matrix(rng):
    """A calibration table: error rate 10^(-q/10) moved by up to a fifth per cycle, unequal substitutions."""
    q = np.arange(256)[:, None]
    err = np.clip(10.0 ** (-q / 10.0), 1e-6, 0.74) * rng.uniform(0.8, 1.0 / 0.8, (256, 256))
    err = np.minimum(err, 0.75)
    share = rng.uniform(0.5, 1.5, (256, 256, 4, 4))
    for t in range(4):
        share[:, :, t, t] = 0.0
    pm = err[:, :, None, None] * share / share.sum(-1, keepdims=True)
    for t in range(4):
        pm[:, :, t, t] = 1.0 - err
    return np.ascontiguousarray(pm.reshape(-1))


def _flags(case):
    return {k: case[k] for k in ("refine_mode", "rank_sum_mode", "transition_dominant", "is_monoploid") if case.get(k)}


def _draw_reads(case, rng):
    """Reads of one chromosome for the window interface: position sorted, one in ten trimmed, 3 % with two hits, a het
    site every 1,000 bases."""
    n_sites, L = case["sites"], case["read"]
    n = max(1, int(case["depth"] * n_sites / L))
    ref = rng.integers(0, 4, n_sites).astype(np.uint8)
    alt = ref.copy()
    het = rng.random(n_sites) < 1e-3
    alt[het] ^= 3
    pos = np.sort(rng.integers(0, n_sites - L - 1, n)).astype(np.int32)
    length = np.where(rng.random(n) < 0.1, rng.integers(max(1, 3 * L // 4), L + 1, n), L).astype(np.int32)
    hit = np.where(rng.random(n) < 0.03, 2, 1).astype(np.int32)
    rev = rng.random(n) < 0.5
    at = pos[:, None].astype(np.int64) + np.arange(L)[None, :]
    base = np.where((rng.random(n) < 0.5)[:, None], ref[at], alt[at])
    qual = np.clip(np.rint(rng.normal(30.0, 7.0, (n, L))), 2, 40).astype(np.uint8)
    wrong = rng.random((n, L)) < 10.0 ** (-qual / 10.0)
    base = np.where(wrong, (base + 1 + rng.integers(0, 3, (n, L))) & 3, base).astype(np.uint8)
    return {"ref": ref, "pos": pos, "length": length, "hit": hit, "rev": rev, "base": base, "qual": qual}


def _draw_records(case, rng):
    """Observation records of sites, 256 slots each: base, quality, cycle and strand of mostly one base, one site in a
    hundred nearly full."""
    n, depth = case["sites"], case["depth"]
    counts = np.clip(rng.poisson(rng.gamma(4.0, depth / 4.0, n)), 0, 256).astype(np.int32)
    deep = rng.random(n) < 0.01
    counts[deep] = rng.integers(200, 257, int(deep.sum()))
    total = int(counts.sum())
    site = np.repeat(np.arange(n), counts)
    slot = np.arange(total) - np.repeat(np.cumsum(counts) - counts, counts)
    base = rng.integers(0, 4, n)[site]
    off = rng.random(total) < 0.03
    base[off] = rng.integers(0, 4, int(off.sum()))
    q = np.clip(np.rint(rng.normal(30.0, 7.0, total)), 2, 40).astype(np.int64)
    cycle, strand = rng.integers(0, 100, total), rng.integers(0, 2, total)
    word = (base << 23) | ((64 - q) << 17) | (cycle << 9) | (strand << 8) | 1
    return {"counts": counts, "site": site, "slot": slot, "word": word.astype(np.int64)}


def _context(pm, **kw):
    L = gsnp_amd.lib()
    gsnp_amd.check(L.gsnp_device_init(0))
    p = gsnp_amd.params(**kw)
    ctx = ctypes.c_void_p()
    gsnp_amd.check(L.gsnp_create(ctypes.byref(p), pm.ctypes.data, ctypes.byref(ctx)))
    return ctx


def prepare(case, seed):
    s = _State(case)
    kind, L = s.kind, gsnp_amd.lib()
    rng = np.random.default_rng(seed)
    if kind == "sorted":
        s.ctx = _context(_p_matrix(rng), read_length=100)
        d = _draw_records(case, rng)
        flat = torch.full((case["sites"] * 256,), -1, dtype=torch.int32, device="cuda")
        flat[torch.from_numpy(d["site"] * 256 + d["slot"]).cuda()] = torch.from_numpy(d["word"]).to(torch.int32).cuda()
        s.records = flat.view(case["sites"], 256)
        s.counts = torch.from_numpy(d["counts"]).cuda()
        s.lk = torch.empty((case["sites"], 10), dtype=torch.float64, device="cuda")
        return s
    if kind == "windows":
        s.ctx = _context(_p_matrix(rng), read_length=case["read"])
        d = _draw_reads(case, rng)
        codes = d["ref"]
        gsnp_amd.check(L.gsnp_set_chromosome(s.ctx, b"chr1", codes.ctypes.data, len(codes), None, None, 0))
        seq = np.frombuffer(b"ACTG", np.uint8)[d["base"]]
        qual = (d["qual"] + 64).astype(np.uint8)
        strand = np.where(d["rev"], ord("-"), ord("+")).astype(np.uint8)
        len_hit = ((d["length"] << 16) | d["hit"]).astype(np.int32)
        rb = gsnp_amd.ReadBatch(len(d["pos"]), case["read"], d["pos"].ctypes.data, len_hit.ctypes.data, strand.ctypes.data,
                                seq.ctypes.data, qual.ctypes.data)
        gsnp_amd.check(L.gsnp_load_reads(s.ctx, ctypes.byref(rb)))
        s.starts = [int(x) for x in np.searchsorted(d["pos"], np.arange(0, case["sites"] + gsnp_amd.WIN, gsnp_amd.WIN))]
        n = case["sites"]
        s.out = {"lk10": _pinned(10 * n, torch.float64), "base1": _pinned(n), "base2": _pinned(n), "type1": _pinned(n),
                 "q_cns": _pinned(n, torch.int32), "depth": _pinned(n, torch.int32)}
        return s
    s.job = gsnp_amd.Job(synth=(case["config"], seed, case["scale"]), **_flags(case))
    s.ctx = s.job.ctx
    s.lens = [s.job.info(i)[1] for i in range(len(s.job))]
    n = _room(case)
    if sum(s.lens) > n:
        raise ValueError("the sample holds more sites than its buffers")
    if kind == "rows":
        s.text = _pinned(ROW_ROOM * n)
    elif kind == "calls":
        s.out = {"base1": _pinned(n), "base2": _pinned(n), "type1": _pinned(n), "q_cns": _pinned(n, torch.int32)}
        if case.get("rank_sum_mode"):
            s.out["rank_sum"] = _pinned(n, torch.float64)
    elif kind == "columns":
        s.chunks = np.zeros(CHUNK_ROOM * n + (1 << 18), np.uint8)
        s.sizes = np.zeros((WINDOW_ROOM, 5), np.int64)
        s.used = s.windows = 0

        def take(user, chrom, start, sites, chunk, size):
            if s.windows >= WINDOW_ROOM:
                return 1
            for f in range(5):
                if s.used + size[f] > s.chunks.size:
                    return 1
                ctypes.memmove(s.chunks.ctypes.data + s.used, chunk[f], size[f])
                s.used += size[f]
                s.sizes[s.windows, f] = size[f]
            s.windows += 1
            return 0

        s.take = gsnp_amd.CHUNK_FN(take)
    elif kind in ("adjoint", "span"):
        s.pm = _p_matrix(rng)
        s.log_het = math.log(1e-3) + 0.1 * rng.standard_normal()
        s.adj = Adjoint(s.job) if kind == "adjoint" else None
    elif kind == "counts":
        s.job.select(0)
    elif kind == "decode":
        s.tmp = tempfile.TemporaryDirectory(prefix="cases_")
        s.prefix = Path(s.tmp.name) / "sample"
        s.job.write(s.prefix, compress=True, batched=32)
        s.text = np.zeros(ROW_ROOM * n, np.uint8)
        s.job.close()
        s.job = s.ctx = None
    return s


# ---- one pass ----------------------------------------------------------------


def _spans(length, per):
    step = per * gsnp_amd.WIN
    return [(a, min(step, length - a)) for a in range(0, length, step)]


def _results(ctx, out, at, n):
    """Per-site results of the last call into the caller's arrays from site `at` on."""
    w = gsnp_amd.WindowOut()
    for k, v in out.items():
        width = 10 if k == "lk10" else 1
        setattr(w, k, v.data_ptr() + at * width * v.element_size())
    gsnp_amd.check(gsnp_amd.lib().gsnp_window_results(ctx, n, ctypes.byref(w)))


def run(s):
    L, check, case = gsnp_amd.lib(), gsnp_amd.check, s.case
    if s.kind == "rows":
        at, nb = 0, ctypes.c_uint64()
        for i, length in enumerate(s.lens):
            s.job.select(i)
            for a, n in _spans(length, case["per"]):
                check(L.gsnp_batched_call(s.ctx, a, n, 1, None))
                check(L.gsnp_fetch_text(s.ctx, ctypes.cast(s.text.data_ptr() + at, ctypes.c_char_p), s.text.numel() - at,
                                        ctypes.byref(nb)))
                at += nb.value
        return s.text
    if s.kind == "calls":
        at = 0
        for i, length in enumerate(s.lens):
            s.job.select(i)
            for a, n in _spans(length, case["per"]):
                check(L.gsnp_batched_call(s.ctx, a, n, 0, None))
                _results(s.ctx, s.out, at, n)
                at += n
        return s.out
    if s.kind == "columns":
        s.used = s.windows = 0
        for i in range(len(s.lens)):
            s.job.select(i)
            check(L.gsnp_job_columns_to(s.job.h, case["per"], s.take, None, None))
        return {"chunks": s.chunks, "sizes": s.sizes}
    if s.kind == "windows":
        check(L.gsnp_window_init(s.ctx, 0))
        for w, a in enumerate(range(0, case["sites"], gsnp_amd.WIN)):
            n = min(gsnp_amd.WIN, case["sites"] - a)
            check(L.gsnp_window_update(s.ctx, s.starts[w], s.starts[w + 1], None))
            check(L.gsnp_window_likelihood(s.ctx, n))
            check(L.gsnp_window_posterior(s.ctx, n))
            _results(s.ctx, s.out, a, n)
            check(L.gsnp_window_recycle(s.ctx))
        return s.out
    if s.kind == "sorted":
        check(L.gsnp_sort_likelihood_noalloc(s.ctx, s.records.data_ptr(), s.counts.data_ptr(), case["sites"],
                                             s.lk.data_ptr()))
        return {"records": s.records, "lk10": s.lk}
    if s.kind == "adjoint":
        out = s.adj.eval(s.pm, s.log_het, site_terms=case["site_terms"])
        return dict(zip(("loglik", "grad", "grad_het", "sites"), out))
    if s.kind == "span":
        s.adj = Adjoint(s.job)
        return dict(zip(("loglik", "grad", "grad_het"), s.adj.eval(s.pm, s.log_het)))
    if s.kind == "counts":
        counts = np.zeros(64 << 12, np.uint64)
        check(L.gsnp_calib_count(s.ctx, counts.ctypes.data))
        return counts.view(np.int64)
    out = Path(s.tmp.name) / "sample.cns"
    gsnp_amd.decompress(s.prefix, out, device=True)
    with open(out, "rb") as f:
        f.readinto(s.text)
    return s.text


# ---- what a pass cannot do without -------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "sorted":
        rec = case["sites"] * case["depth"]
        return {"bytes": 8 * rec + 84 * case["sites"], "flops": 10 * rec}  # records sorted in place, sums out
    if kind == "windows":
        rec = case["sites"] * case["depth"]
        return {"bytes": rec + 12 * rec / case["read"] + (1 + 80 + 3 + 4 + 4) * case["sites"], "flops": 10 * rec}
    sites = SITES[case["config"]] * case["scale"]
    rec = sites * DEPTH[case["config"]]
    reads = rec + 12 * rec / READ[case["config"]] + sites  # a byte per base, 12 per read, a reference code per site
    if kind == "rows":
        return {"bytes": reads + ROW_BYTES * sites, "flops": 10 * rec}
    if kind == "calls":
        return {"bytes": reads + (15 if case.get("rank_sum_mode") else 7) * sites, "flops": 10 * rec}
    if kind == "columns":
        return {"bytes": reads + 6 * sites, "flops": 10 * rec}
    if kind == "adjoint":  # a key per record, a prior row per site, the table in and the gradient out
        return {"bytes": 4 * rec + 4 * sites + 2 * 64 * 4096 * 8, "flops": 20 * rec}
    if kind == "span":
        return {"bytes": reads + 2 * 64 * 4096 * 8, "flops": 20 * rec}
    if kind == "counts":
        return {"bytes": reads + 64 * 4096 * 8, "flops": rec}
    return {"bytes": (6 + ROW_BYTES) * sites, "flops": 0}


# ---- the same outputs in plain 64-bit torch ----------------------------------


def _likelihoods(site, base, qual, cycle, strand, n_sites, pm, pcr=0.5, glob=0.9):
    """Ten log10 likelihoods per site: each observation's quality lowered for the observations of its base before it (in
    base, quality down, cycle, strand order) that repeat its cycle and strand (pcr) or have others (glob)."""
    key = (site << 19) | (base << 17) | ((64 - qual) << 11) | (cycle << 2) | strand
    order = torch.argsort(key, stable=True)
    site, base, qual, cycle, strand = (x[order] for x in (site, base, qual, cycle, strand))
    same = (site << 13) | (base << 11) | (cycle << 2) | strand
    o2 = torch.argsort(same, stable=True)
    s2 = same[o2]
    place = torch.arange(s2.numel(), device=s2.device)
    head = torch.ones_like(s2, dtype=torch.bool)
    head[1:] = s2[1:] != s2[:-1]
    rep = torch.empty_like(place)
    rep[o2] = place - torch.cummax(torch.where(head, place, 0), 0).values
    seg = (site << 2) | base
    new = torch.ones_like(seg, dtype=torch.bool)
    new[1:] = seg[1:] != seg[:-1]
    firsts = torch.cumsum((rep == 0).long(), 0)
    other = firsts - torch.cummax(torch.where(new, firsts, 0), 0).values
    x = torch.log10(qual.double()) + rep.double() * math.log10(pcr) + other.double() * math.log10(glob)
    qa = torch.clamp((torch.pow(10.0, x) + 0.5).floor().long(), min=1)
    p = torch.from_numpy(pm).to(site.device).view(256, 256, 4, 4)
    lk = torch.zeros((n_sites, 10), dtype=torch.float64, device=site.device)
    for g, (a1, a2) in enumerate(GENOTYPES):
        lk[:, g].index_add_(0, site, torch.log10(0.5 * p[qa, cycle, a1, base] + 0.5 * p[qa, cycle, a2, base]))
    return lk


def _adjoint_exact(case, s, adj):
    dev = "cuda"
    keys, off, prow = adj.export()
    het, hom = math.exp(s.log_het), 0.0005
    prior = torch.zeros((8, 10), dtype=torch.float64)
    for r in range(8):
        for g, (a, b) in enumerate(GENOTYPES):
            if r < 4:
                prior[r, g] = (1.0 if a == r else hom) if a == b else het if r in (a, b) else het * hom
            else:
                prior[r, g] = (1.0 if a == b else 2 * het) * 0.0625
    ln_prior = torch.log(prior).to(dev)
    mask = torch.tensor([a != b for a, b in GENOTYPES], device=dev)
    p = torch.from_numpy(s.pm).to(dev).view(256, 256, 4, 4)[:64]
    pk = p.permute(0, 1, 3, 2).reshape(-1, 4)  # by q, cycle, obs: the four p over the true base
    table = torch.log(torch.stack([0.5 * pk[:, a] + 0.5 * pk[:, b] for a, b in GENOTYPES], 1))
    weights = torch.zeros((65536, 10), dtype=torch.float64, device=dev)
    terms, dhet = [], 0.0
    off = off.astype(np.int64)
    for a in range(0, adj.n_sites, 250_000):
        b = min(adj.n_sites, a + 250_000)
        k = torch.from_numpy(keys[off[a]:off[b]].astype(np.int64)).to(dev)
        seg = torch.repeat_interleave(torch.arange(b - a, device=dev), torch.from_numpy(np.diff(off[a:b + 1])).to(dev))
        v = torch.zeros((b - a, 10), dtype=torch.float64, device=dev)
        v.index_add_(0, seg, table[k])
        v += ln_prior[torch.from_numpy(prow[a:b].astype(np.int64)).to(dev)]
        terms.append(torch.logsumexp(v, 1))
        w = torch.softmax(v, 1)
        dhet += float(w[:, mask].sum())
        weights.index_add_(0, k, w[seg])
    grad = torch.zeros((65536, 4), dtype=torch.float64, device=dev)
    for g, (a, b) in enumerate(GENOTYPES):
        t = pk[:, a] + pk[:, b]
        grad[:, a] += weights[:, g] * pk[:, a] / t
        grad[:, b] += weights[:, g] * pk[:, b] / t
    terms = torch.cat(terms)
    out = {"loglik": float(terms.sum()), "grad": grad.view(64, 256, 4, 4).permute(0, 1, 3, 2).contiguous().cpu().numpy(),
           "grad_het": dhet}
    if case.get("site_terms"):
        out["sites"] = terms.cpu().numpy()
    return out


def exact(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    gpu = lambda x: torch.from_numpy(np.ascontiguousarray(x)).long().cuda()  # noqa: E731
    if kind == "sorted":
        pm = _p_matrix(rng)
        d = _draw_records(case, rng)
        w = gpu(d["word"])
        lk = _likelihoods(gpu(d["site"]), (w >> 23) & 3, 64 - ((w >> 17) & 63), (w >> 9) & 255, (w >> 8) & 1, case["sites"], pm)
        return {"records": None, "lk10": lk}
    if kind == "windows":
        pm = _p_matrix(rng)
        d = _draw_reads(case, rng)
        k = np.arange(case["read"])[None, :]
        on = (k < d["length"][:, None]) & (d["hit"] == 1)[:, None]
        # the caller drops a read that reaches the chromosome's last base: none is drawn there
        i, j = np.nonzero(on)
        cycle = np.where(d["rev"][i], d["length"][i] - 1 - j, j)
        lk = _likelihoods(gpu(d["pos"][i].astype(np.int64) + j), gpu(d["base"][i, j]), gpu(d["qual"][i, j]), gpu(cycle),
                          gpu(d["rev"][i]), case["sites"], pm)
        return {"lk10": lk.reshape(-1).cpu(), "base1": None, "base2": None, "type1": None, "q_cns": None, "depth": None}
    if kind in ("adjoint", "span"):
        s = prepare(case, seed)
        return _adjoint_exact(case, s, s.adj or Adjoint(s.job))
    return None
