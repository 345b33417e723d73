"""The screen that answers gapless pairs from their bytes, against the oracle,
bit for bit: near its conditions' limits (mismatches packed into a word, near
copies on other diagonals, short gaps), at its word edges, with overhanging and
shorter references."""
import random

import numpy as np
import pytest

from test_gpu_sw_lean import check

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    from swift_amd import align
    return align


LENGTHS = [15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 79, 80, 81, 111, 112, 150, 255, 256, 257,
           300, 319, 320]


def screen_pairs(rnd, n, qmax):
    qs, rs = [], []
    lengths = [x for x in LENGTHS if x <= qmax]
    for i in range(n):
        ql = rnd.choice(lengths)
        kind = rnd.randrange(8)
        unit = rnd.choice((1, 2, 3, 5, 16, 31, 32, 33, 50))
        rl = rnd.randint(1, 480) if kind == 0 else min(480, ql + rnd.randint(0, 180))
        if kind == 1:  # tandem: equal copies on other diagonals
            u = bytes(rnd.choice(b"ACGT") for _ in range(unit))
            reg = bytearray((u * (rl // unit + 1))[:rl])
        else:
            reg = bytearray(rnd.choice(b"ACGT") for _ in range(rl))
        if kind == 2 and rl > 80:  # a second copy of a stretch, a few bases off
            a, m = rnd.randint(0, rl - 41), rnd.randint(20, 40)
            b = rnd.randint(0, rl - m)
            reg[b:b + m] = reg[a:a + m][:rl - b]
        o = rnd.randint(-20, max(0, rl - ql) + 20) if kind == 3 else rnd.randint(0, max(0, rl - ql))
        q = bytearray(rnd.choice(b"ACGT") for _ in range(ql))
        for k in range(ql):
            if 0 <= o + k < rl:
                q[k] = reg[o + k]
        if kind == 4:  # mismatches packed together, at an end as often as not
            a = rnd.choice((0, ql - 8, rnd.randint(0, ql - 8)))
            for k in rnd.sample(range(a, a + 8), rnd.randint(1, 6)):
                q[k] = rnd.choice([c for c in b"ACGT" if c != q[k]])
        if kind == 5:  # a gap either way, anywhere
            p, d = rnd.randint(0, ql - 1), rnd.randint(1, 12)
            q = (q[:p] + q[p + d:] if i % 2 else q[:p] + reg[:d] + q[p:])[:ql] or q
        rate = rnd.choice((0, 0, 0.01, 0.03, 0.1))
        for k in range(len(q)):
            if rnd.random() < rate:
                q[k] = rnd.choice(b"ACGT")
        if kind == 6:
            q[rnd.randrange(len(q))] = rnd.choice(b"Na")
        if kind == 7:
            reg[rnd.randrange(rl)] = rnd.choice(b"NRacgt")
        if i % 9 == 0:
            reg = reg.lower()
        qs.append(bytes(q))
        rs.append(bytes(reg))
    return qs, rs


# the default scoring; a gap as cheap as a mismatch; one that outweighs many; no
# mismatch allowed in a word; extending dearer than opening; the packed forms
SCORINGS = [(2, -1, -10, -1), (1, -1, -1, -1), (1, -1, -63, -1), (1, -30, -3, -2),
            (3, -2, -2, -63), (5, -4, -12, -2), (6, -1, -11, -1), (1, -1, -16, -1)]


@pytest.mark.parametrize("sc", SCORINGS)
@pytest.mark.parametrize("rows", [0, -1])
def test_screen(A, orc, sc, rows):
    """rows 0: the kernel ahead of the bins; -1: inside the small call's."""
    rnd = random.Random(sum(sc) * 7 + rows)
    qs, rs = screen_pairs(rnd, 6000, 320)
    before = A.get_coarse_rows()
    try:
        A.set_coarse_rows(rows)
        got = A.sw_batch(qs, rs, A.Scoring(*sc))
    finally:
        A.set_coarse_rows(before)
    check(got, orc.sw_batch(qs, rs, *sc, nthreads=8))


def test_screen_takes_reads(A, orc):
    """Reads with a substitution or two beside their places leave the bins."""
    rnd = random.Random(2)
    qs, rs = [], []
    for i in range(2000):
        reg = bytes(rnd.choice(b"ACGT") for _ in range(300))
        o = rnd.randint(0, 150)
        q = bytearray(reg[o:o + 150])
        for k in rnd.sample(range(150), i % 3):
            q[k] = rnd.choice(b"ACGT")
        qs.append(bytes(q))
        rs.append(reg)
    before = A.get_coarse_rows()
    try:
        A.set_coarse_rows(0)
        got = A.sw_batch(qs, rs)
        assert A.batch_stats()["ntasks16"] <= 3
    finally:
        A.set_coarse_rows(before)
    check(got, orc.sw_batch(qs, rs, nthreads=8))


@pytest.mark.parametrize("ql,rl", [(16, 40), (100, 300), (143, 200), (320, 480)])
def test_screen_plain(A, orc, ql, rl):
    """The plain path's packed route: the screen, and the sweep of its list;
    references that end early."""
    rnd = random.Random(ql)
    qs, rs = screen_pairs(rnd, 4200, 320)
    for i in range(len(qs)):
        reg = rs[i][:rl].ljust(rl if i % 3 else 1, b"G")
        o = rnd.randint(0, max(0, len(reg) - ql))
        q = reg[o:o + ql].upper().ljust(ql, b"C") if i % 2 else qs[i].ljust(ql, b"T")[:ql]
        qs[i], rs[i] = q, reg
    got = A.align_sequences(qs, rs, ql, rl)
    sc, st, en, al, qc, rc = orc.sw_batch(qs, rs, nthreads=8)
    check(got, (sc.astype(np.float32), st, en, al, qc, rc))
