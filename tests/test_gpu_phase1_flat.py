"""The flat mapping tier (reads of at most 320 k-mers, 32-bit cluster ids)
against the oracle: read lengths on both sides of its rounds and of its limit,
strands on both sides of its hit capacity, more sequences than a wave has
lanes, indexes with and without the bucket bitmap."""
import random

import pytest

from test_gpu_phase1 import check_strands

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    from swift_amd import search
    return search


def sample(rnd, seqs, lengths, orc):
    """Mutated stretches of the sequences on either strand, with other bytes."""
    reads = []
    for n in lengths:
        s = rnd.choice([q for q in seqs if len(q) > n + 1] or [bytes(rnd.choices(b"ACGT", k=n + 2))])
        p = rnd.randrange(len(s) - n)
        r = bytearray(s[p:p + n])
        for i in range(n):
            if rnd.random() < 0.02:
                r[i] = rnd.choice(b"ACGTNacgtR")
        reads.append(bytes(r) if rnd.random() < 0.5 else orc.revcomp(bytes(r)))
    return reads


# k = 4: 256 buckets, every one filled (no bitmap); k = 12 on 60 kbp: few are;
# k = 13: past the bitmap's size
@pytest.mark.parametrize("k,nseq,total", [(4, 3, 3000), (12, 5, 60000), (12, 127, 60000),
                                          (13, 66, 30000)])
@pytest.mark.parametrize("max_hits", [1, 4])
def test_flat_lengths(S, orc, k, nseq, total, max_hits):
    rnd = random.Random(100 * k + nseq)
    seqs = [bytes(rnd.choices(b"ACGT", k=rnd.randint(1, 2 * total // nseq))) for _ in range(nseq)]
    for nq in (128, 320, 321):  # the longest read picks the tier
        edge = [0, 1, k - 1, k, k + 1] + [max(1, b + d) for b in (16, 63, 64, 128, 192, 319)
                                          for d in (-1, 0, 1)]
        lengths = [n for n in edge if n <= nq + k - 1] + [nq + k - 1]
        reads = sample(rnd, seqs, lengths * 3, orc)
        got = S.Index.from_sequences(seqs, k, 100000).map_reads(reads, max_hits)
        check_strands(orc.Index(seqs, k, 100000), reads, got, max_hits, orc)


@pytest.mark.parametrize("copies", [1, 3, 32, 33, 40])
def test_flat_hit_capacity(S, orc, copies):
    """A unit repeated `copies` times at every phase of the tuple grid: 8 tuples
    of a read hit each copy, so 32 copies make 256 hits and 33 pass them on."""
    rnd = random.Random(copies)
    k = 12
    unit = bytes(rnd.choices(b"ACGT", k=8 * k))
    seqs = [b"".join(unit + bytes(rnd.choices(b"ACGT", k=k)) for _ in range(copies)),
            bytes(rnd.choices(b"ACGT", k=5000))]
    reads = [unit, unit[:50], unit[5:], unit + unit[:20], orc.revcomp(unit)]
    got = S.Index.from_sequences(seqs, k, 1000).map_reads(reads, 3)
    want = orc.Index(seqs, k, 1000)
    assert want.map_query(unit, 3, orc.TIE_FIRST)[2] >= 8 * copies
    check_strands(want, reads, got, 3, orc)


def test_index_bucket_sizes(S, orc):
    """Buckets of every size a sort network takes, and on both sides of the
    one-thread, one-wave and workgroup sorts, spread over three sequences."""
    rnd = random.Random(9)
    k = 8
    sizes = list(range(1, 41)) + [63, 64, 65, 1023, 1024, 1025, 2049]
    kmers = rnd.sample(range(4 ** k), len(sizes))
    grid = [m for m, n in zip(kmers, sizes) for _ in range(n)]
    rnd.shuffle(grid)
    text = ["".join("ACGT"[(m >> (2 * i)) & 3] for i in range(k)) for m in grid]
    cut = len(text) // 3
    seqs = ["".join(text[a:b]).encode() for a, b in ((0, cut), (cut, 2 * cut), (2 * cut, None))]
    for thr in (5000, 33):
        got = S.Index.from_sequences(seqs, k, thr).arrays()
        want = orc.Index(seqs, k, thr).arrays()
        for key in ("start", "count", "actual", "refIdx", "refPos"):
            assert (got[key] == want[key]).all(), (thr, key)
