"""The lean sweeps (scorings whose exits' penalties fit a byte) against the
oracle, bit for bit: at the edges of their rule, at every row class's first
and last query length, with wildcards next to padding rows and columns."""
import random

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    from swift_amd import align
    return align


def edge_pairs(rnd, n, qmax, rmax):
    """Queries at and beside multiples of 16 and 64, mutated from their
    regions, with N on either side, lower case, and ends of unequal length."""
    qs, rs = [], []
    for i in range(n):
        ql = min(qmax, max(1, rnd.choice((16, 64)) * rnd.randint(0, 20) + rnd.randint(-1, 1)))
        rl = rnd.randint(1, rmax) if i % 4 else rmax
        reg = bytearray(rnd.choice(b"ACGT") for _ in range(rl))
        o = rnd.randint(0, max(0, rl - ql))
        q = reg[o:o + ql] + bytes(rnd.choice(b"ACGT") for _ in range(ql - len(reg[o:o + ql])))
        for k in range(ql):
            if rnd.random() < 0.04:
                q[k] = rnd.choice(b"ACGTNacgt")
        if i % 3 == 0:  # a gap either way
            p = rnd.randint(0, ql - 1)
            d = rnd.randint(1, 9)
            q = (q[:p] + q[p + d:] if i % 2 else q[:p] + bytes(b"ACGTACGTA"[:d]) + q[p:])[:ql] or q
        for k in range(rl):
            if rnd.random() < 0.03:
                reg[k] = rnd.choice(b"NNnacgt" if i % 5 else b"NRYk")
        e = min(rl, o + len(q))  # wildcards right after the query's last row
        reg[e:e + 6] = b"N" * len(reg[e:e + 6])
        qs.append(bytes(q))
        rs.append(bytes(reg))
    return qs, rs


def check(got, want):
    sc, st, en, al, qc, rc = want
    assert np.array_equal(got.score, sc)
    assert np.array_equal(got.start, st) and np.array_equal(got.end, en)
    assert np.array_equal(got.length, al)
    assert got.qry_cons == qc and got.ref_cons == rc


# scoring, longest query: the default; each limit of the rule (match - mismatch
# 31, penalties of 63) and one past it; scores on both sides of the packed
# forms' limits (960 - match, 2016 - match)
EDGES = [((2, -1, -10, -1), 320), ((1, -30, -63, -1), 320), ((1, -31, -10, -1), 200),
         ((3, -2, -2, -63), 316), ((3, -2, -64, -2), 316), ((3, -1, -5, -2), 320),
         ((30, -1, -63, -63), 30), ((30, -1, -63, -63), 32), ((5, -4, -12, -4), 190),
         ((5, -4, -12, -4), 200), ((1, -1, -1, -2), 100), ((6, -5, -13, -3), 320),
         ((30, -1, -63, -63), 66), ((30, -1, -63, -63), 67), ((7, -3, -9, -2), 290)]


@pytest.mark.parametrize("form", ["rows", "coarse", "wide", "int32"])
@pytest.mark.parametrize("sc,qmax", EDGES)
def test_batch_lean_edges(A, orc, sc, qmax, form):
    rnd = random.Random(1000 * qmax + sc[0])
    n = 700 if form != "coarse" else 4100
    qs, rs = edge_pairs(rnd, n, qmax, 480 if form != "coarse" else 130)
    rows, tune = A.get_coarse_rows(), A.get_tuning()
    try:
        A.set_coarse_rows(0 if form in ("rows", "int32") else 1)
        if form == "int32":
            A.set_tuning(allow_int16=False, walk_deferred=True)
        got = A.sw_batch(qs, rs, A.Scoring(*sc))
    finally:
        A.set_coarse_rows(rows)
        A.set_tuning(tune["waves_per_cu"], tune["allow_int16"], tune["walk_deferred"])
    check(got, orc.sw_batch(qs, rs, *sc, nthreads=8))


# the packed rule's limits (match - mismatch 15, penalties of 31) and one past each
@pytest.mark.parametrize("sc", [(14, -1, -31, -1), (1, -14, -31, -31), (1, -15, -10, -1),
                                (1, -1, -32, -1), (2, -1, -16, -16), (2, -1, -5, -32)])
@pytest.mark.parametrize("rows", [0, -1])
def test_batch_packed_edges(A, orc, sc, rows):
    rnd = random.Random(sum(sc))
    qs, rs = edge_pairs(rnd, 1500, min(320, 900 // sc[0]), 400)
    before = A.get_coarse_rows()
    try:
        A.set_coarse_rows(rows)
        got = A.sw_batch(qs, rs, A.Scoring(*sc))
    finally:
        A.set_coarse_rows(before)
    check(got, orc.sw_batch(qs, rs, *sc, nthreads=8))


# rows a lane capped at the longest query's, also where a call says less than that
@pytest.mark.parametrize("qmax,said", [(100, 100), (161, 161), (177, 100), (33, 1)])
def test_batch_coarse_cap(A, orc, qmax, said):
    rnd = random.Random(qmax)
    qs, rs = edge_pairs(rnd, 4300, qmax, 200)
    before = A.get_coarse_rows()
    try:
        A.set_coarse_rows(1)
        b = A.PairBatch(qs, rs)
        b.maxq = said
        b.run()
    finally:
        A.set_coarse_rows(before)
    check(b.results(), orc.sw_batch(qs, rs, nthreads=8))
