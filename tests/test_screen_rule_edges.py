"""The screen's rule at the edges of its conditions, and that it answers pairs at
all: mismatches in a word up to what a gap costs and one past it, words as long
as K, scorings that leave it nothing."""
import random

import pytest

from test_screen_rule import screen


def near_pairs(rnd, n, lengths, rates):
    qs, rs = [], []
    for _ in range(n):
        ql = rnd.choice(lengths)
        r = bytes(rnd.choice(b"ACGT") for _ in range(ql + rnd.randint(0, 60)))
        o = rnd.randint(-4, len(r) - ql + 4)
        rate = rnd.choice(rates)
        q = bytes(r[o + k] if 0 <= o + k < len(r) and rnd.random() >= rate
                  else rnd.choice(b"ACGT") for k in range(ql))
        qs.append(q)
        rs.append(r)
    return qs, rs


def answered(orc, qs, rs, m, x, g, e):
    """How many pairs the rule answers, each as the oracle's matrix does."""
    sc, st, en, al, _, _ = orc.sw_batch(qs, rs, m, -x, -g, -e, nthreads=4)
    n = 0
    for i, (q, r) in enumerate(zip(qs, rs)):
        got = screen(q, r, m, x, g)
        assert got is None or got == (sc[i], st[i], en[i], al[i]), (i, m, x, g, e)
        n += got is not None
    return n


# scoring and the least share of near copies answered: the default; K = 16, a
# word's rows, and one past it (the last word only); K = 1; a gap cheaper than
# one mismatch; no word long enough
@pytest.mark.parametrize("sc,share", [((2, 1, 10, 1), 0.5), ((1, 1, 16, 1), 0.15),
                                      ((1, 1, 17, 1), 0.05), ((5, 4, 12, 2), 0.2),
                                      ((3, 1, 3, 1), 0.0), ((1, 3, 4, 1), 0.0),
                                      ((1, 1, 48, 1), None)])
def test_answers(orc, sc, share):
    rnd = random.Random(sum(sc))
    qs, rs = near_pairs(rnd, 800, (16, 31, 32, 47, 48, 63, 64, 79, 80, 110, 150),
                        (0, 0, 0.01, 0.03))
    n = answered(orc, qs, rs, *sc)
    assert n == 0 if share is None else n > share * len(qs), n


@pytest.mark.parametrize("m,x,e", [(2, 1, 3), (1, 1, 2), (1, 2, 4), (3, 5, 2), (5, 4, 1)])
def test_mismatches_in_a_word(orc, m, x, e):
    """e mismatches of one word against gaps that cost one more than they could
    win, as much, and less."""
    rnd = random.Random(m * 100 + x * 10 + e)
    qs, rs = [], []
    while len(qs) < 60:
        r = bytes(rnd.choice(b"ACGT") for _ in range(120))
        q = bytearray(r[10:106])
        w = rnd.randrange(3)
        for k in rnd.sample(range(32 * w, 32 * w + 32), e):
            q[k] = rnd.choice([c for c in b"ACGT" if c != q[k]])
        qs.append(bytes(q))
        rs.append(r)
    gap = (m + x) * e
    assert answered(orc, qs, rs, m, x, gap + 1, 1) >= 55  # a chance copy beside it may show
    assert answered(orc, qs, rs, m, x, gap, 1) == 0
    assert answered(orc, qs, rs, m, x, gap - 1, 1) == 0
