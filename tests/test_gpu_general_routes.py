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


class NoAlloc:
    """The no-allocation call over its own buffers."""

    def __init__(self, n, ql, rl, sc):
        from swift_amd.device import DeviceBuffer
        self.n, self.ql, self.rl, self.sc, self.cl = n, ql, rl, sc, ql + rl + 2
        self.q, self.r = DeviceBuffer(n * (ql + 1)), DeviceBuffer(n * (rl + 1))
        self.out = ([DeviceBuffer(4 * n) for _ in range(4)]
                    + [DeviceBuffer(self.cl * n) for _ in range(2)])

    def load(self, qs, rs):
        for buf, seqs, width in ((self.q, qs, self.ql), (self.r, rs, self.rl)):
            a = np.zeros((self.n, width + 1), np.uint8)
            for i, s in enumerate(seqs):
                a[i, :len(s)] = np.frombuffer(s, np.uint8)
            buf.upload(a)

    def run(self, stream=None):
        from swift_amd._lib import check as ok
        from swift_amd._lib import lib
        ok(lib().swift_align_sequences_noalloc(
            self.q.cptr, self.r.cptr, self.ql, self.rl, *(C.c_float(x) for x in self.sc),
            *(x.cptr for x in self.out), self.n, stream))

    def check(self, want):
        from swift_amd._lib import check as ok
        from swift_amd._lib import lib
        ok(lib().swift_device_synchronize())
        for x, w in zip(self.out, want[:4]):
            assert np.array_equal(x.download(np.int32 if x is not self.out[0] else np.float32,
                                             self.n), w)
        for x, w in zip(self.out[4:], want[4:]):
            rows = x.download(np.uint8, self.cl * self.n).reshape(self.n, self.cl)
            assert [s.tobytes().split(b"\0")[0] for s in rows] == list(w)


# chunks of the 64 MiB array: two of the packed route, three of the general one,
# the waves of the wave route over and over
@pytest.mark.parametrize("n,ql,rl,sc", [(6000, 100, 300, (2, -1, -10, -1)),
                                        (1600, 100, 300, GENERAL),
                                        (5000, 300, 320, (2, -1, -10, -1))])
def test_noalloc_chunks(orc, n, ql, rl, sc):
    qs, rs = edge_pairs(random.Random(n), n, ql, rl)
    qs = [q.ljust(ql, b"G")[:ql] for q in qs]
    call = NoAlloc(n, ql, rl, sc)
    call.load(qs, rs)
    call.run()
    call.check(orc.sw_batch(qs, rs, *sc, nthreads=8))


@pytest.mark.parametrize("n,ql,rl,sc", [(6000, 100, 300, (2, -1, -10, -1)),
                                        (300, 100, 300, (2, -1, -10, -1)),
                                        (800, 100, 300, GENERAL)])
def test_noalloc_replays(orc, n, ql, rl, sc):
    """Captured once; every replay is over other pairs, with eager calls between."""
    from swift_amd._lib import lib
    from swift_amd.device import Stream
    lib()
    hip = C.CDLL("libamdhip64.so")
    sets = []
    for seed in range(3):
        qs, rs = edge_pairs(random.Random(seed), n, ql, rl)
        qs = [q.ljust(ql, b"G")[:ql] for q in qs]
        sets.append((qs, rs, orc.sw_batch(qs, rs, *sc, nthreads=8)))
    call, other, st = NoAlloc(n, ql, rl, sc), NoAlloc(n, ql, rl, sc), Stream()
    graph, run = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(st.cptr, 0) == 0
    call.run(st.cptr)
    assert hip.hipStreamEndCapture(st.cptr, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, 0) == 0
    for i in (0, 1, 2, 0):
        qs, rs, want = sets[i]
        call.load(qs, rs)
        assert hip.hipGraphLaunch(run, st.cptr) == 0
        st.synchronize()
        call.check(want)
        other.load(*sets[(i + 1) % 3][:2])
        other.run()
        other.check(sets[(i + 1) % 3][2])
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0


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
