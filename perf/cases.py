"""Work that a program using this library has it do, as cases to time.

Every case goes through the public entry points: the batched and the plain
Smith-Waterman calls on pairs resident on the device, read mapping, the
phase-1 -> phase-2 pipeline, the serving loop, and a whole run from a
reference in host memory (index, map, align).  Sizes come from the benchmark
configurations (bench.py, swift_amd/synth.py) and the tests.

Inputs are made on the GPU from the seed: uniform or repeat-carrying genomes,
reads sampled from them at the configurations' error rates, pairs whose query
is a mutated copy of a stretch of its region.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from swift_amd import search
from swift_amd._lib import check, lib
from swift_amd.align import PairBatch, Scoring
from swift_amd.device import DeviceBuffer
from swift_amd.serve import Server

BASES = b"ACGT"
DEFAULT = {"match": 2, "mismatch": -1, "gap_open": -10, "gap_ext": -1}


def listed():
    return [
        # a handful of candidates aligned on demand: launches and latency
        _batch("batch-64", 64, 50, 300, 20, 180),
        # one serving-sized batch of mixed read lengths
        _batch("batch-8k", 8_000, 50, 300, 20, 180),
        # the batched benchmark: a million uneven pairs
        _batch("batch-1m", 1_000_000, 36, 250, 20, 200),
        # long queries near the batched limits, references with ambiguity
        # codes in places, and a scoring of the user's own
        _batch("batch-iupac", 100_000, 101, 319, 20, 160, iupac=0.05, match=5, mismatch=-4,
               gap_open=-12, gap_ext=-2),
        # the drop-in call (one fixed stride): a small one, and every
        # candidate window of a large read set
        _plain("plain-256", 256, 143, 253),
        _plain("plain-100k", 100_000, 100, 300),
        # phase 1 alone: both strands of every read, 50 Mbp reference
        _reads("map-105k", "map", 50_000_000, 24, "tandem", 105_000, 100, 100),
        # the whole pipeline: 1 Mbp and 1,000 reads; 50 Mbp and 105,000
        # reads; 3.1 Gbp and one 250,000-read batch of its stream
        _reads("align-1k", "align", 1_000_000, 1, "none", 1_000, 100, 100, sub=0.02),
        _reads("align-105k", "align", 50_000_000, 24, "tandem", 105_000, 100, 100),
        _reads("align-250k", "align", 3_100_000_000, 25, "dispersed", 250_000, 150, 150),
        # a service's requests of mixed sizes and read lengths, in flight
        # together over a resident index
        _reads("serve-24", "serve", 50_000_000, 24, "tandem", 24, 50, 300, sub=0.015),
        # one command-line run: index the reference, map and align a read set
        _reads("oneshot-20k", "oneshot", 50_000_000, 24, "tandem", 20_000, 100, 100),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("batch", "batch", "plain", "map", "align", "align", "serve", "oneshot"))
    if kind == "batch":
        qmin = rng.randint(30, 200)
        c = _batch("", log_int(20, 400_000), qmin, rng.randint(qmin, 300), 20,
                   rng.randint(20, 180))
        if rng.random() < 0.3:
            c.update(iupac=rng.choice((0.01, 0.1)), match=rng.choice((1, 3, 5)),
                     mismatch=rng.choice((-4, -3, -1)), gap_open=-rng.randint(3, 16),
                     gap_ext=-rng.randint(1, 3))
    elif kind == "plain":
        q = rng.randint(30, 300)
        c = _plain("", log_int(20, 60_000), q, q + rng.randint(20, 200))
    else:
        genome = log_int(1_000_000, 200_000_000)
        lo = rng.randint(40, 200)
        n = log_int(4, 40) if kind == "serve" else log_int(50, 100_000)
        c = _reads("", kind, genome, rng.randint(1, 25),
                   rng.choice(("none", "tandem", "dispersed")), n, lo, rng.randint(lo, 300),
                   sub=rng.choice((0.005, 0.01, 0.03)))
    del c["name"]
    return c


def _batch(name, n, qmin, qmax, dmin, dmax, iupac=0.0, **scoring):
    return {"name": name, "kind": "batch", "n": n, "qmin": qmin, "qmax": qmax, "dmin": dmin,
            "dmax": dmax, "iupac": iupac, **DEFAULT, **scoring}


def _plain(name, n, qlen, rlen):
    return {"name": name, "kind": "plain", "n": n, "qlen": qlen, "rlen": rlen, **DEFAULT}


def _reads(name, kind, genome, nseq, repeats, n, lmin, lmax, sub=0.01):
    """n: reads, or for "serve" requests of log-uniform 1..4096 reads."""
    return {"name": name, "kind": kind, "genome": genome, "nseq": nseq, "repeats": repeats,
            "n": n, "lmin": lmin, "lmax": lmax, "sub": sub, "k": 12, "threshold": 1000,
            "max_hits": 3, **DEFAULT}


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _letters(codes):
    return torch.tensor(list(BASES), dtype=torch.uint8, device="cuda")[codes.long()]


def _random_codes(g, n, gc=0.41):
    """Base codes (A C G T = 0..3) at the given GC content."""
    out = torch.empty(n, dtype=torch.uint8, device="cuda")
    at = int(round(1000 * (1 - gc)))
    for a in range(0, n, 1 << 28):
        m = min(1 << 28, n - a)
        x = torch.randint(0, 1000, (m,), generator=g, device="cuda", dtype=torch.int16)
        # the two low-order letters of each class alternate with the value's parity
        out[a:a + m] = torch.where(x < at, 3 * (x & 1), 1 + (x & 1)).to(torch.uint8)
    return out


def _spread(lens):
    """(row of each element, its index within the row) of ragged rows."""
    row = torch.repeat_interleave(torch.arange(len(lens), device="cuda"), lens)
    first = torch.cumsum(lens, 0) - lens
    return row, torch.arange(int(lens.sum()), device="cuda") - first[row]


def _mutated(g, codes, rate):
    """Substitutions by one of the other three bases."""
    hit = torch.rand(codes.shape, generator=g, device="cuda") < rate
    step = torch.randint(1, 4, codes.shape, generator=g, device="cuda", dtype=torch.uint8)
    return torch.where(hit, (codes + step) & 3, codes)


def _genome(g, total, repeats):
    """Base codes: "tandem" puts 5 % of the bases in tandem arrays of period
    2..50, "dispersed" 45 % in diverged copies of 300..6000-base families."""
    codes = _random_codes(g, total)
    # one copy per stretch of the genome, so that no two overlap
    if repeats == "tandem":
        stretch = 10_920
        n = total // stretch
        period = torch.randint(2, 51, (n,), generator=g, device="cuda")
        span = period * torch.randint(3, 40, (n,), generator=g, device="cuda")
        units = _random_codes(g, n * 50)
        row, k = _spread(span)
        at = _place(g, n, stretch, span)
        codes[at[row] + k] = units[row * 50 + k % period[row]]
    elif repeats == "dispersed":
        stretch = 7_000
        flen = torch.randint(300, 6001, (1000,), generator=g, device="cuda")
        ffirst = torch.cumsum(flen, 0) - flen
        family = _random_codes(g, int(flen.sum()))
        for a in range(0, total // stretch, 50_000):  # a part at a time: 8 bytes a base
            n = min(50_000, total // stretch - a)
            which = torch.randint(0, 1000, (n,), generator=g, device="cuda")
            at = a * stretch + _place(g, n, stretch, flen[which])
            row, k = _spread(flen[which])
            codes[at[row] + k] = _mutated(g, family[ffirst[which][row] + k], 0.15)
    return codes


def _place(g, n, stretch, span):
    """A start within each of n stretches that leaves room for its span."""
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    return torch.arange(n, device="cuda") * stretch + (u * (stretch - span).double()).long()


def _sequences(g, total, nseq):
    """Offsets and lengths of nseq sequences of uneven lengths, back to back."""
    share = 0.2 + torch.rand(nseq, generator=g, device="cuda", dtype=torch.float64)
    lens = (share / share.sum() * total).long()
    lens[-1] += total - lens.sum()
    return (torch.cumsum(lens, 0) - lens), lens


def _sample_reads(g, codes, off, lens, n, lmin, lmax, sub):
    """Reads from uniform places of either strand, 5 % of them random bases:
    letters, offsets and lengths in host memory."""
    rl = torch.randint(lmin, lmax + 1, (n,), generator=g, device="cuda")
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    which = torch.searchsorted(torch.cumsum(lens, 0).double() / int(lens.sum()), u)
    which = which.clamp_(max=len(lens) - 1)
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    at = off[which] + (u * (lens[which] - rl).double()).long()
    reverse = torch.rand(n, generator=g, device="cuda") < 0.5
    stray = torch.rand(n, generator=g, device="cuda") < 0.05
    row, k = _spread(rl)
    src = torch.where(reverse[row], at[row] + rl[row] - 1 - k, at[row] + k)
    c = codes[src]
    c = torch.where(reverse[row], 3 - c, c)  # complement: A-T, C-G
    c = torch.where(stray[row], _random_codes(g, len(c)), c)
    c = _letters(_mutated(g, c, sub))
    pad = torch.zeros(8, dtype=torch.uint8, device="cuda")
    roff = torch.cumsum(rl, 0) - rl
    return (torch.cat([c, pad]).cpu().numpy(), roff.cpu().numpy(),
            rl.to(torch.int32).cpu().numpy())


def _pairs(g, qlen, rlen, sub, indel, iupac):
    """Regions of random bases and queries copied from within them, with
    substitutions and for some a one-base insertion or deletion.  Returns
    query and region letters (ragged, back to back)."""
    n = len(qlen)
    region = _random_codes(g, int(rlen.sum()), gc=0.5)
    rfirst = torch.cumsum(rlen, 0) - rlen
    shift = (torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
             * (rlen - qlen + 1)).long()
    event = torch.rand(n, generator=g, device="cuda") < indel * qlen
    insert = torch.rand(n, generator=g, device="cuda") < 0.5
    place = (torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * qlen).long()
    row, k = _spread(qlen)
    past = event[row] & (k >= place[row])
    k2 = torch.where(past, torch.where(insert[row], k - 1, k + 1), k)
    k2 = torch.minimum(k2.clamp(min=0), (rlen - shift)[row] - 1)
    query = _mutated(g, region[rfirst[row] + shift[row] + k2], sub)
    letters = _letters(region)
    if iupac > 0:
        # ambiguity codes at a few columns of some regions
        bad = torch.rand(n, generator=g, device="cuda") < iupac
        rrow, _ = _spread(rlen)
        spot = bad[rrow] & (torch.rand(len(rrow), generator=g, device="cuda") < 0.02)
        codes = torch.tensor(list(b"RYKMSWNN"), dtype=torch.uint8, device="cuda")
        pick = torch.randint(0, 8, (len(rrow),), generator=g, device="cuda")
        letters = torch.where(spot, codes[pick], letters)
    return _letters(query), letters


def _pair_lengths(g, case):
    n = case["n"]
    if case["kind"] == "plain":
        return (torch.full((n,), case["qlen"], device="cuda"),
                torch.full((n,), case["rlen"], device="cuda"))
    qlen = torch.randint(case["qmin"], case["qmax"] + 1, (n,), generator=g, device="cuda")
    extra = torch.randint(case["dmin"], case["dmax"] + 1, (n,), generator=g, device="cuda")
    return qlen, qlen + extra


def _pair_inputs(case, seed):
    g = _generator(seed)
    qlen, rlen = _pair_lengths(g, case)
    q, r = _pairs(g, qlen, rlen, 0.018, 0.002, case.get("iupac", 0.0))
    return qlen, rlen, q, r


def _scoring(case):
    return Scoring(case["match"], case["mismatch"], case["gap_open"], case["gap_ext"])


def _request_sizes(n):
    """Log-uniform over 1..4096 reads."""
    return [int(4096 ** ((i + 0.5) / n)) for i in range(n)]


# ---------------------------------------------------------- device outputs
class _Memory:
    def __init__(self, buf, dtype, count):
        self.keep = buf
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": np.dtype(dtype).str,
                                         "data": (buf.ptr, False), "version": 2}


def _view(buf, dtype, count):
    """A DeviceBuffer as a tensor, without a copy."""
    return torch.as_tensor(_Memory(buf, dtype, count), device="cuda")


def _zeroed(nbytes):
    b = DeviceBuffer(nbytes)
    b.zero()
    return b


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return _prepare_batch(case, seed)
    if kind == "plain":
        return _prepare_plain(case, seed)
    g = _generator(seed)
    codes = _genome(g, case["genome"], case["repeats"])
    off, lens = _sequences(g, case["genome"], case["nseq"])
    if kind == "serve":
        sizes = _request_sizes(case["n"])
        sizes = [sizes[i] for i in torch.randperm(len(sizes), generator=g, device="cuda").tolist()]
    else:
        sizes = [case["n"]]
    reads = [_sample_reads(g, codes, off, lens, m, case["lmin"], case["lmax"], case["sub"])
             for m in sizes]
    text = torch.empty_like(codes)
    for a in range(0, len(codes), 1 << 28):
        text[a:a + (1 << 28)] = _letters(codes[a:a + (1 << 28)])
    del codes
    text = text.cpu().numpy()
    off, lens = off.cpu().numpy(), lens.cpu().numpy()
    s = {"kind": kind, "case": case, "scoring": _scoring(case)}
    if kind == "oneshot":
        return {**s, "text": text, "off": off, "lens": lens, "reads": reads[0]}
    s["index"] = search.Index.from_packed(text, off, lens, case["k"], case["threshold"])
    mh = case["max_hits"]
    if kind == "serve":
        s["server"] = Server(s["index"], nslots=4, mem_budget=32 << 30, max_batch_reads=8192,
                             max_read_len=case["lmax"], max_hits=mh, scoring=s["scoring"])
        return {**s, "requests": reads}
    rb = s["reads"] = search.ReadBatch.from_packed(*reads[0], max_read_len=case["lmax"])
    if kind == "map":
        ns = 2 * rb.n
        kinds = {"ref": (np.int8, ns * mh), "shift": (np.int32, ns * mh),
                 "pos": (np.int32, ns * mh), "nbest": (np.int32, ns), "nbiggest": (np.int32, ns),
                 "nhits": (np.int32, ns)}
        s["bufs"] = {f: _zeroed(np.dtype(t).itemsize * c) for f, (t, c) in kinds.items()}
        s["out"] = {f: _view(s["bufs"][f], t, c) for f, (t, c) in kinds.items()}
    else:
        rec = s["records"] = search.RecordBuffers(2 * rb.n * mh, rb.max_len)
        for b in rec.bufs.values():
            b.zero()
        cap = rec.capacity
        s["out"] = {f: _view(rec.bufs[f], np.int32, cap) for f in search.I32_FIELDS}
        s["out"]["nrecords"] = _view(rec.bufs["nrecords"], np.int32, 1)
        s["out"]["ref_distance"] = _view(rec.bufs["ref_distance"], np.int64, cap)
        for f in ("qry_cons", "ref_cons"):
            s["out"][f] = _view(rec.bufs[f], np.uint8, cap * rec.stride)
    return s


def _strings_stride(case):
    if case["kind"] == "plain":
        return case["qlen"] + case["rlen"] + 2
    return (2 * case["qmax"] + case["dmax"] + 2 + 3) // 4 * 4


def _prepare_batch(case, seed):
    qlen, rlen, q, r = _pair_inputs(case, seed)
    pad = torch.zeros(8, dtype=torch.uint8, device="cuda")
    host = [x.cpu().numpy() for x in (
        torch.cat([q, pad]), torch.cumsum(qlen, 0) - qlen, qlen, torch.cat([r, pad]),
        torch.cumsum(rlen, 0) - rlen, rlen)]
    b = PairBatch.from_arrays(*host)
    size = case["n"] * _strings_stride(case)  # room for the longest pairs' strings
    b.qc, b.rc = DeviceBuffer(size), DeviceBuffer(size)
    for buf in (b.score, b.start, b.end, b.alen, b.qc, b.rc):
        buf.zero()
    out = {f: _view(getattr(b, f), np.int32, b.n) for f in ("score", "start", "end", "alen")}
    for f in ("qc", "rc"):
        out[f] = _view(getattr(b, f), np.uint8, size)
    return {"kind": "batch", "case": case, "scoring": _scoring(case), "batch": b, "out": out}


def _prepare_plain(case, seed):
    n, ql, rl = case["n"], case["qlen"], case["rlen"]
    _, _, q, r = _pair_inputs(case, seed)
    fixed = []
    for x, width in ((q, ql), (r, rl)):  # stride width + 1, NUL terminated
        rows = torch.zeros(n, width + 1, dtype=torch.uint8, device="cuda")
        rows[:, :width] = x.view(n, width)
        fixed.append(DeviceBuffer.from_array(rows.cpu().numpy()))
    width = _strings_stride(case)
    bufs = {f: _zeroed(4 * n) for f in ("score", "start", "end", "alen")}
    bufs.update({f: _zeroed(width * n) for f in ("qc", "rc")})
    out = {f: _view(b, np.uint8, width * n) if f in ("qc", "rc") else
           _view(b, np.float32 if f == "score" else np.int32, n) for f, b in bufs.items()}
    return {"kind": "plain", "case": case, "scoring": _scoring(case), "q": fixed[0],
            "r": fixed[1], "bufs": bufs, "out": out}


# --------------------------------------------------------------------- run
def run(s):
    kind, case, sc = s["kind"], s["case"], s["scoring"]
    if kind == "batch":
        s["batch"].run(sc)
        return s["out"]
    if kind == "plain":
        b = s["bufs"]
        check(lib().swift_align_sequences(
            s["q"].cptr, s["r"].cptr, case["qlen"], case["rlen"], C.c_float(sc.match),
            C.c_float(sc.mismatch), C.c_float(sc.gap_open), C.c_float(sc.gap_ext),
            b["score"].cptr, b["start"].cptr, b["end"].cptr, b["alen"].cptr, b["qc"].cptr,
            b["rc"].cptr, case["n"], None))
        return s["out"]
    mh = case["max_hits"]
    if kind == "map":
        rb, b = s["reads"], s["bufs"]
        check(lib().swift_map_reads(
            s["index"]._h, rb.seq.cptr, rb.off.cptr, rb.len.cptr, rb.n, rb.max_len, mh,
            b["ref"].cptr, b["shift"].cptr, b["pos"].cptr, b["nbest"].cptr, b["nbiggest"].cptr,
            b["nhits"].cptr, None))
        return s["out"]
    if kind == "align":
        s["index"].align_batch(s["reads"], s["records"], mh, sc)
        return s["out"]
    if kind == "serve":
        ids = [s["server"].submit_packed(*r) for r in s["requests"]]
        return _columns([s["server"].result(i, strings=False)[0] for i in ids],
                        2 * mh * sum(len(r[2]) for r in s["requests"]))
    index = search.Index.from_packed(s["text"], s["off"], s["lens"], case["k"],
                                     case["threshold"])
    rb = search.ReadBatch.from_packed(*s["reads"], max_read_len=case["lmax"])
    rec = search.RecordBuffers(2 * rb.n * mh, rb.max_len)
    index.align_batch(rb, rec, mh, sc)
    out = _columns([rec.results(strings=False)], rec.capacity)
    index.close()
    return out


def _columns(parts, capacity):
    """The records of one request after another, in arrays of the most there can be."""
    out = {}
    for f in search.I32_FIELDS + ("ref_distance",):
        out[f] = np.zeros(capacity, parts[0].cols[f].dtype)
        at = 0
        for p in parts:
            out[f][at:at + p.n] = p.cols[f]
            at += p.n
    out["records"] = sum(p.n for p in parts)
    return out


# -------------------------------------------------------------------- work
def work(case):
    """Bytes: every input read and every output written once.  Operations: 16
    integer operations a Smith-Waterman cell."""
    if case["kind"] == "plain":
        n, q, r = case["n"], case["qlen"], case["rlen"]
        return {"bytes": n * (q + r + 16 + 2 * (q + 1)), "flops": 16.0 * n * q * r}
    if case["kind"] == "batch":
        n, a, b = case["n"], case["qmin"], case["qmax"]
        q, d = (a + b) / 2, (case["dmin"] + case["dmax"]) / 2
        cells = n * (q * q + ((b - a + 1) ** 2 - 1) / 12 + q * d)
        return {"bytes": n * (2 * q + d + 40 + 16 + 2 * (q + 1)), "flops": 16.0 * cells}
    n = case["n"]
    if case["kind"] == "serve":
        n = sum(_request_sizes(n))
    length = (case["lmin"] + case["lmax"]) / 2
    kmers = 2 * n * max(length - case["k"] + 1, 1)
    tuples = case["genome"] / case["k"]
    per_kmer = tuples / 4 ** case["k"]
    # phase 1: the reads, 8 bytes a bucket, 4 bytes a hit, the hits reported
    best = n * (1 + min(case["max_hits"], kmers / (2 * n) * per_kmer))
    bytes_ = n * (length + 12) + kmers * (8 + 4 * per_kmer) + 9 * best
    if case["kind"] == "map":
        return {"bytes": bytes_, "flops": kmers}
    # phase 2: a 300-base window a record, the record and its strings
    bytes_ += best * (length + 300 + 60 + 2 * length)
    if case["kind"] == "oneshot":
        bytes_ += case["genome"] + 8 * tuples + 8 * 4 ** case["k"]
    return {"bytes": bytes_, "flops": 16.0 * best * length * 300}


# ------------------------------------------------------------------- exact
def exact(case, seed):
    """Smith-Waterman of the pair cases by anti-diagonals in 64-bit integers.
    The read cases' outputs are picks, positions and whole scores: None."""
    if case["kind"] not in ("batch", "plain"):
        return None
    qmax = case.get("qmax", case.get("qlen"))
    rmax = case["rlen"] if case["kind"] == "plain" else qmax + case["dmax"]
    if case["n"] * qmax * (qmax + rmax) > 3e10:  # about 20 seconds
        return None
    qlen, rlen, q, r = _pair_inputs(case, seed)
    n = case["n"]
    if case["kind"] == "plain":
        stride = torch.full((n,), case["qlen"] + case["rlen"] + 2, device="cuda")
    else:
        stride = (qlen + rlen + 2 + 3) // 4 * 4
    first = torch.cumsum(stride, 0) - stride
    size = n * _strings_stride(case)
    qc, rc = (torch.zeros(size, dtype=torch.uint8, device="cuda") for _ in range(2))
    cols = [torch.zeros(n, dtype=torch.int64, device="cuda") for _ in range(4)]
    part = max(1, int(1.5e9 // (qmax * (qmax + rmax))))
    q_at, r_at = torch.cumsum(qlen, 0) - qlen, torch.cumsum(rlen, 0) - rlen
    for a in range(0, n, part):
        p = slice(a, min(n, a + part))
        got = _exact_part(_padded(q, q_at[p], qlen[p]), _padded(r, r_at[p], rlen[p]), qlen[p],
                          rlen[p], case, first[p], qc, rc)
        for c, x in zip(cols, got):
            c[p] = x
    score = cols[0].double() if case["kind"] == "plain" else cols[0].to(torch.int32)
    return {"score": score, "start": cols[1].to(torch.int32), "end": cols[2].to(torch.int32),
            "alen": cols[3].to(torch.int32), "qc": qc, "rc": rc}


def _padded(x, first, lens):
    k = torch.arange(int(lens.max()), device="cuda")[None, :]
    at = torch.minimum(first[:, None] + k, first[:, None] + lens[:, None] - 1)
    return torch.where(k < lens[:, None], x[at], torch.zeros_like(x[at]))


def _exact_part(q, r, qlen, rlen, case, first, qc, rc):
    n, Q = q.shape
    R = r.shape[1]
    rows = torch.arange(Q, device="cuda")
    N = ord("N")
    h1, h2 = (torch.zeros(n, Q + 1, dtype=torch.int64, device="cuda") for _ in range(2))
    d1 = torch.zeros(n, Q + 1, dtype=torch.uint8, device="cuda")
    dirs = torch.zeros(Q + R, n, Q, dtype=torch.uint8, device="cuda")
    best = torch.zeros(n, dtype=torch.int64, device="cuda")
    span = (Q + 1) * (R + 1)
    for d in range(Q + R - 1):  # cells (i, d - i), 0-based; h1[:, i + 1] is row i's last value
        col = d - rows
        on = (col >= 0)[None, :] & (col[None, :] < rlen[:, None]) & (rows[None, :] < qlen[:, None])
        rb = r[:, col.clamp(0, R - 1)]
        same = (q == rb) | (q == N) | (rb == N)
        diag = h2[:, :-1] + torch.where(same, case["match"], case["mismatch"])
        up = h1[:, :-1] + torch.where(d1[:, :-1] == 2, case["gap_ext"], case["gap_open"])
        left = h1[:, 1:] + torch.where(d1[:, 1:] == 1, case["gap_ext"], case["gap_open"])
        key = torch.maximum(torch.maximum(4 * diag + 3, 4 * up + 2), 4 * left + 1).clamp_(min=0)
        key = torch.where(on, key, torch.zeros_like(key))
        dirs[d] = (key & 3).to(torch.uint8)
        cell = (key >> 2) * span + (span - 1 - (rows * (R + 1) + col.clamp(min=0)))[None, :]
        best = torch.maximum(best, torch.where(key >= 4, cell, 0).amax(1))
        h2 = h1.clone()
        # cells outside the matrix keep their border value: 0, a start
        h1[:, 1:] = key >> 2
        d1[:, 1:] = dirs[d]
    score = best // span
    at = span - 1 - best % span
    live = score > 0
    i = torch.where(live, at // (R + 1), 0)
    j = torch.where(live, at % (R + 1), 0)
    start, alen = torch.zeros_like(score), torch.zeros_like(score)
    ncol = torch.zeros_like(score)
    who = torch.arange(n, device="cuda")
    for _ in range(Q + R):
        if not bool(live.any()):
            break
        c = dirs[(i + j).clamp(min=0), who, i.clamp(min=0)]
        live = live & (c != 0)
        w = who[live]
        o = first[w] + alen[w]
        gap = torch.full_like(o, ord("-"), dtype=torch.uint8)
        qc[o] = torch.where(c[w] == 1, gap, q[w, i[w]])
        rc[o] = torch.where(c[w] == 2, gap, r[w, j[w]])
        start[w] = j[w] + 1
        alen[w] += 1
        ncol[w] += (c[w] != 2).long()
        i[w] -= (c[w] & 2 != 0).long()
        j[w] -= (c[w] & 1 != 0).long()
        live = live & (i >= 0) & (j >= 0)
    return score, start, start + ncol - 1, alen
