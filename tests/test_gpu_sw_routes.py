"""Which way the batched and the plain path take a call, where the pairs are not
the related ones that the screen answers: its list, and the lines between the
routes."""
import random
import time

import numpy as np
import pytest

from test_gpu_sw_lean import check

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    from swift_amd import align
    return align


def pairs(seed, n, qmin, qmax, extra, related):
    """Random regions; queries copied from them, or random bases."""
    rng = np.random.default_rng(seed)
    letters = np.frombuffer(b"ACGT", np.uint8)
    qs, rs = [], []
    for ql in rng.integers(qmin, qmax + 1, n):
        reg = letters[rng.integers(0, 4, ql + extra)]
        o = int(rng.integers(0, extra + 1))
        q = reg[o:o + ql] if related else letters[rng.integers(0, 4, ql)]
        qs.append(q.tobytes())
        rs.append(reg.tobytes())
    return qs, rs


def least(f, reps=25):
    best = 1e9
    for _ in range(reps):
        t = time.perf_counter()
        f()
        best = min(best, time.perf_counter() - t)
    return best


def test_list_of_unrelated_pairs(A, orc):
    """The screen leaves every pair: its list costs a call less than the row
    classes, which have none, save (it was 1.27 of their time with an atomic a
    wave on the list's length, and is 0.99)."""
    qs, rs = pairs(1, 20_000, 100, 100, 100, False)
    b = A.PairBatch(qs, rs)
    before = A.get_coarse_rows()
    took = {}
    try:
        for rows in (-1, 1):
            A.set_coarse_rows(rows)
            b.run()
            check(b.results(), orc.sw_batch(qs, rs, nthreads=8))
            took[rows] = least(b.run)
    finally:
        A.set_coarse_rows(before)
    assert took[-1] < 1.15 * took[1], took


@pytest.mark.parametrize("related", [True, False])
def test_one_launch_by_the_pairs_left(A, orc, related):
    """A call within the one launch's line: taken by it where the screen answers
    the pairs, handed on to the row classes where it leaves too many."""
    n = 26_000
    qs, rs = pairs(2, n, 30, 60, 60, related)
    # one pair of three rows a lane: two pairs a workgroup
    (qs[5],), (rs[5],) = pairs(3, 1, 170, 170, 20, False)
    got = A.sw_batch(qs, rs)
    tasks = A.batch_stats()["ntasks16"]
    check(got, orc.sw_batch(qs, rs, nthreads=8))
    assert tasks == n // 2 if related else tasks < n // 4
