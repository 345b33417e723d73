"""The screen's rule (swift_amd/csrc/sw_screen.hpp) restated over plain arrays
and held against the oracle's full matrices: wherever its conditions hold, the
best alignment is the one it names.  Pairs with copies of stretches on near
diagonals, small alphabets, overhanging ends; gaps as cheap as a mismatch and
dearer than many."""
import random

import numpy as np
import pytest


def screen(q, r, m, x, g):
    """(score, start, end, length) where every word of one diagonal has few
    mismatches and every word of every other has at least K; else None."""
    ql, rl = len(q), len(r)
    if ql < 16 or rl < 8:
        return None
    k, nw = -(-g // m), (ql + 31) // 32
    cuts = [32 * i for i in range(nw)] + [ql]
    if nw > 1 and ql - 32 * (nw - 1) < 16:
        del cuts[-2]
    ref = np.zeros(rl + 2 * ql, np.uint8)
    ref[ql:ql + rl] = np.frombuffer(r, np.uint8)
    at = np.arange(ql)[None, :] + np.arange(ql + rl)[:, None]  # by diagonal + ql
    miss = (ref[at] != np.frombuffer(q, np.uint8)[None, :]).astype(np.int32)
    upto = np.concatenate([np.zeros((len(miss), 1), np.int32), np.cumsum(miss, 1)], 1)
    words = upto[:, cuts[1:]] - upto[:, cuts[:-1]]
    live = np.nonzero((words < k).any(1))[0]
    if len(live) != 1 or ((m + x) * words[live[0]] >= g).any():
        return None
    best = run = first = row = best_first = 0
    for i, miss_i in enumerate(miss[live[0]]):
        run += -x if miss_i else m
        if run < 0:
            run, first = 0, i + 1
        elif run > best:
            best, row, best_first = run, i, first
    diag = int(live[0]) - ql
    return best, best_first + diag + 1, row + diag + 1, row - best_first + 1


@pytest.mark.parametrize("seed", range(12))
def test_rule(orc, seed):
    rnd = random.Random(seed)
    m, x, g, e = rnd.choice((1, 2, 3, 5)), rnd.randint(1, 6), rnd.randint(1, 20), rnd.randint(1, 4)
    qs, rs = [], []
    for _ in range(600):
        ql = rnd.choice((16, 17, 31, 32, 33, 47, 48, 63, 64, 70, 96, 110))
        rl = rnd.randint(max(8, ql - 15), ql + 60)
        letters = rnd.choice((b"ACGT", b"ACGT", b"ACG", b"AC"))
        r = bytearray(rnd.choice(letters) for _ in range(rl))
        o = rnd.randint(-6, max(0, rl - ql) + 6)
        q = bytearray(r[o + k] if 0 <= o + k < rl else rnd.choice(letters) for k in range(ql))
        for _ in range(rnd.randint(0, 5)):
            a = rnd.randint(0, ql - 4)
            if rnd.random() < 0.5:  # a stretch's copy on a near diagonal
                s = rnd.choice((-6, -3, -2, -1, 1, 2, 3, 5, 9))
                for k in range(a, min(ql, a + rnd.randint(3, 24))):
                    if 0 <= o + k + s < rl:
                        r[o + k + s] = q[k]
                for k in range(ql):
                    if 0 <= o + k < rl and rnd.random() < 0.97:
                        q[k] = r[o + k]
            else:
                for k in range(a, a + rnd.randint(1, 4)):
                    q[k] = rnd.choice(letters)
        qs.append(bytes(q))
        rs.append(bytes(r))
    sc, st, en, al, _, _ = orc.sw_batch(qs, rs, m, -x, -g, -e, nthreads=4)
    for i in range(len(qs)):
        got = screen(qs[i], rs[i], m, x, g)
        assert got is None or got == (sc[i], st[i], en[i], al[i]), (i, m, x, g, e)
