"""The ways past the one launch of small calls: captured row classes, the wide
form, fused and deferred walks of coarse classes, chunks of the no-allocation
call, and the walks of a lane a pair."""
import ctypes as C
import random

import numpy as np
import pytest

from parity_util import assert_records_match
from test_gpu_graph import same
from test_gpu_sw_lean import check, edge_pairs
from test_gpu_sw_routes import pairs

pytestmark = pytest.mark.gpu

GENERAL = (2, -1, -64, -1)  # outside lean_scoring: the general sweeps


@pytest.fixture(scope="module")
def A():
    from swift_amd import align
    return align


# row classes of every height; coarse ones (from 4,096 pairs: 700 slots of 6)
@pytest.mark.parametrize("rows,slots", [(0, 320), (1, 700)])
def test_graph_of_row_classes(A, orc, rows, slots):
    """Every replay, with eager work and synchronisations between, gives the
    eager pipeline's records and the oracle's."""
    from swift_amd import search, synth
    rng = np.random.default_rng(rows)
    seqs = [synth.random_bases(rng, n, 0.41) for n in (250_000, 120_000)]
    ix = search.Index.from_sequences([s.tobytes() for s in seqs], 12, 1000)
    oix = orc.Index([s.tobytes() for s in seqs], 12, 1000)
    sets = [synth.sample_reads(rng, seqs, n, length, 0.015, 0.003)[0]
            for length, n in ((100, slots - 20), (150, 200), (60, slots - 1))]
    before = A.get_coarse_rows()
    try:
        A.set_coarse_rows(rows)
        g = search.PipelineGraph(ix, slots, 150, 3)
    finally:
        A.set_coarse_rows(before)
    try:
        for rep, reads in enumerate(sets + [sets[0]]):
            got = g.run(reads)
            padded = list(reads) + [b""] * (g.slots - len(reads))
            same(got, ix.align_reads(padded, 3, max_read_len=150), rep)
            assert got.n > 0
            assert_records_match(got, orc.pipeline(oix, reads, 3), rep)
    finally:
        g.close()


@pytest.mark.parametrize("deferred", [False, True])
@pytest.mark.parametrize("sc", [(2, -1, -10, -1), GENERAL])
def test_coarse_walks(A, orc, deferred, sc):
    qs, rs = edge_pairs(random.Random(17), 4500, 300, 400)
    tune, rows = A.get_tuning(), A.get_coarse_rows()
    try:
        A.set_tuning(tune["waves_per_cu"], True, deferred)
        A.set_coarse_rows(1)
        got = A.sw_batch(qs, rs, A.Scoring(*sc))
        assert A.batch_stats()["nrerun"] > 0
    finally:
        A.set_tuning(tune["waves_per_cu"], tune["allow_int16"], tune["walk_deferred"])
        A.set_coarse_rows(rows)
    check(got, orc.sw_batch(qs, rs, *sc, nthreads=8))


def test_wide_form_limits(A, orc):
    """The largest call of the wide form, whose scorings are the general ones:
    the longest pairs beside short ones."""
    rnd = random.Random(29)
    qs, rs = edge_pairs(rnd, 4095, 320, 480)
    got = A.sw_batch(qs, rs, A.Scoring(*GENERAL))
    assert A.batch_stats()["ntasks16"] == 2048
    check(got, orc.sw_batch(qs, rs, *GENERAL, nthreads=8))


def noalloc(qs, rs, ql, rl, sc):
    from swift_amd._lib import check as ok
    from swift_amd._lib import lib
    from swift_amd.device import DeviceBuffer
    n, cl = len(qs), ql + rl + 2

    def fixed(seqs, width):
        a = np.zeros((n, width + 1), np.uint8)
        for i, s in enumerate(seqs):
            a[i, :len(s)] = np.frombuffer(s, np.uint8)
        return DeviceBuffer.from_array(a)

    q, r = fixed(qs, ql), fixed(rs, rl)
    b = [DeviceBuffer(4 * n) for _ in range(4)] + [DeviceBuffer(cl * n) for _ in range(2)]
    ok(lib().swift_align_sequences_noalloc(q.cptr, r.cptr, ql, rl, *(C.c_float(x) for x in sc),
                                           *(x.cptr for x in b), n, None))
    ok(lib().swift_device_synchronize())
    cols = [x.download(t, n) for x, t in zip(b, (np.float32, np.int32, np.int32, np.int32))]
    return cols + [x.download(np.uint8, cl * n).reshape(n, cl) for x in b[4:]]


# chunks of the 64 MiB array: two of the packed route, three of the general one,
# the waves of the wave route over and over
@pytest.mark.parametrize("n,ql,rl,sc", [(6000, 100, 300, (2, -1, -10, -1)),
                                        (1600, 100, 300, GENERAL),
                                        (5000, 300, 320, (2, -1, -10, -1))])
def test_noalloc_chunks(orc, n, ql, rl, sc):
    qs, rs = edge_pairs(random.Random(n), n, ql, rl)
    qs = [q.ljust(ql, b"G")[:ql] for q in qs]
    s, st, en, al, qc, rc = orc.sw_batch(qs, rs, *sc, nthreads=8)
    got = noalloc(qs, rs, ql, rl, sc)
    for a, b in zip(got, (s.astype(np.float32), st, en, al)):
        assert np.array_equal(a, b)
    for a, want in zip(got[4:], (qc, rc)):
        assert [x.tobytes().split(b"\0")[0] for x in a] == list(want)


# the first calls whose walks take a lane a pair: a class of the batched path,
# the plain path's packed and general routes
def test_lane_walks_batch(A, orc):
    qs, rs = pairs(4, 41_500, 33, 48, 20, False)
    before = A.get_coarse_rows()
    try:
        A.set_coarse_rows(0)
        got = A.sw_batch(qs, rs)
    finally:
        A.set_coarse_rows(before)
    check(got, orc.sw_batch(qs, rs, nthreads=8))


@pytest.mark.parametrize("n,sc", [(131_080, (2, -1, -10, -1)), (16_390, GENERAL)])
def test_lane_walks_plain(A, orc, n, sc):
    qs, rs = pairs(5, n, 30, 30, 12, False)
    got = A.align_sequences(qs, rs, 30, 42, A.Scoring(*sc))
    s, st, en, al, qc, rc = orc.sw_batch(qs, rs, *sc, nthreads=8)
    check(got, (s.astype(np.float32), st, en, al, qc, rc))
