"""The plain path's one-launch and packed routes against the oracle, at the
sizes where they change."""
import random

import numpy as np
import pytest

from test_gpu_sw_lean import check, edge_pairs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    from swift_amd import align
    return align


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
