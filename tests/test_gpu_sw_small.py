"""The one-launch forms of small calls (batched and plain) and the plain path's
packed route against the oracle, at the sizes where they change."""
import random

import numpy as np
import pytest

from test_gpu_sw_lean import check, edge_pairs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    from swift_amd import align
    return align


# pairs: one; the last with a pair a wave, the first with two (an odd count);
# past one turn of the persistent waves; queries: each rows-per-lane count
@pytest.mark.parametrize("n,qmax,rmax", [(1, 320, 480), (1024, 64, 300), (1025, 65, 97),
                                         (2049, 160, 250), (300, 192, 480), (77, 320, 30),
                                         (9001, 128, 200)])
def test_small_batch(A, orc, n, qmax, rmax):
    rnd = random.Random(n)
    qs, rs = edge_pairs(rnd, n, qmax, rmax)
    if n > 10:  # empty sequences: no strings, an empty alignment
        qs[3], rs[5] = b"", b""
    got = A.sw_batch(qs, rs)
    if n > 100:
        assert A.batch_stats()["nrerun"] > 0  # references with R, Y or k
    if n > 10:
        assert got.end[3] == got.end[5] == -1 and got.length[3] == got.length[5] == 0
    check(got, orc.sw_batch(qs, rs, nthreads=8))


def test_small_batch_longer_than_said(A, orc):
    """maxq and maxr below the pairs' own lengths: the call still aligns them."""
    rnd = random.Random(5)
    qs, rs = edge_pairs(rnd, 200, 300, 400)
    b = A.PairBatch(qs, rs)
    b.maxq, b.maxr = 90, 120
    b.run()
    check(b.results(), orc.sw_batch(qs, rs, nthreads=8))


# the wave route (any lengths) and the packed one from 4,096 pairs: rows 1, a
# full and a ragged class, the longest; references near their limits
@pytest.mark.parametrize("n,ql,rl", [(1, 1, 1), (130, 64, 63), (4096, 1, 40), (4097, 16, 33),
                                     (4103, 145, 200), (4096, 320, 90), (40, 65, 2500),
                                     (60, 476, 600), (60, 640, 700), (4100, 30, 1024),
                                     (4100, 30, 1025)])
def test_plain_routes(A, orc, n, ql, rl):
    rnd = random.Random(n + ql)
    qs, rs = edge_pairs(rnd, n, ql, rl)
    qs = [q.ljust(ql, rnd.choice((b"A", b"N", b"c")))[:ql] for q in qs]
    got = A.align_sequences(qs, rs, ql, rl)
    sc, st, en, al, qc, rc = orc.sw_batch(qs, rs, nthreads=8)
    check(got, (sc.astype(np.float32), st, en, al, qc, rc))


@pytest.mark.parametrize("sc,n,ql,rl", [((5, -4, -12, -2), 4099, 201, 260),
                                        ((6, -5, -13, -3), 70, 320, 400),
                                        ((3, -2, -64, -2), 4099, 60, 90)])
def test_plain_scorings(A, orc, sc, n, ql, rl):
    """Packed route with the wider keys, wave route past them, general route."""
    rnd = random.Random(n + ql)
    qs, rs = edge_pairs(rnd, n, ql, rl)
    qs = [q.ljust(ql, b"G")[:ql] for q in qs]
    got = A.align_sequences(qs, rs, ql, rl, A.Scoring(*sc))
    s, st, en, al, qc, rc = orc.sw_batch(qs, rs, *sc, nthreads=8)
    check(got, (s.astype(np.float32), st, en, al, qc, rc))
