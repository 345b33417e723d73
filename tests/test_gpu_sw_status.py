"""Calls of the batched path that do not wait (a serving slot's, a graph's): a
pair too long for them is reported at the next check, once, and the pairs beside
it and the calls after it are answered."""
import ctypes as C
import random

import pytest

from test_gpu_sw_lean import check, edge_pairs

pytestmark = pytest.mark.gpu


class BatchIO(C.Structure):  # swift_amd/csrc/sw_host.hpp
    _fields_ = ([(f, C.c_void_p) for f in ("qseq", "qoff", "qlen", "rseq", "roff", "rlen")]
                + [(f, C.c_int) for f in ("npairs", "maxq", "maxr")]
                + [(f, C.c_void_p) for f in ("score", "start", "end", "alen", "qcons", "rcons",
                                             "cons_off")]
                + [("refs_plain", C.c_int), ("sparse", C.c_int)])


class Scoring(C.Structure):
    _fields_ = [(f, C.c_int) for f in ("match", "mismatch", "gap_open", "gap_ext")]


class Path:
    """The internal calls of one private workspace, on its own stream."""
    NAMES = {"run": "_ZN5swift15sw_batch_run_inEPNS_9WorkspaceERKNS_7BatchIOERKNS_7ScoringEP12ihipStream_t",
             "enqueue": "_ZN5swift19sw_batch_enqueue_inEPNS_9WorkspaceERKNS_7BatchIOERKNS_7ScoringEP12ihipStream_t",
             "reserve": "_ZN5swift16reserve_batch_inEPNS_9WorkspaceEiii",
             "check": "_ZN5swift17sw_batch_check_inEPNS_9WorkspaceEP12ihipStream_t",
             "status": "_ZN5swift18sw_batch_status_inEPNS_9WorkspaceE",
             "new": "_ZN5swift13workspace_newEi", "free": "_ZN5swift14workspace_freeEPNS_9WorkspaceE"}

    def __init__(self, npairs=0, maxq=0, maxr=0):
        from swift_amd._lib import lib
        from swift_amd.device import Stream
        self.f = {k: getattr(lib(), v) for k, v in self.NAMES.items()}
        self.f["new"].restype = C.c_void_p
        self.st = Stream()
        self.w = C.c_void_p(self.f["new"](0))
        if npairs:
            assert self.f["reserve"](self.w, npairs, maxq, maxr) == 0

    def call(self, how, b, sc, sparse=1):
        io = BatchIO(b.q.ptr, b.qo.ptr, b.ql.ptr, b.r.ptr, b.ro.ptr, b.rl.ptr, b.n, b.maxq,
                     b.maxr, b.score.ptr, b.start.ptr, b.end.ptr, b.alen.ptr, b.qc.ptr, b.rc.ptr,
                     b.co.ptr, 0, sparse)
        rc = self.f[how](self.w, C.byref(io), C.byref(Scoring(*sc)), self.st.cptr)
        if rc:
            return rc
        if how == "enqueue":
            return self.f["check"](self.w, self.st.cptr)
        self.st.synchronize()
        return self.f["status"](self.w)

    def close(self):
        self.st.synchronize()
        self.f["free"](self.w)


# lean_packed scorings take the one launch, others the row classes
@pytest.mark.parametrize("how", ["run", "enqueue"])
@pytest.mark.parametrize("sc", [(2, -1, -10, -1), (2, -1, -64, -1)])
@pytest.mark.parametrize("long_q,long_r", [(321, 100), (50, 481)])
def test_too_long_pair_is_reported(orc, how, sc, long_q, long_r):
    from swift_amd import align as A
    qs, rs = edge_pairs(random.Random(long_q), 300, 120, 200)
    good = A.PairBatch(qs, rs)
    bad = A.PairBatch(qs[:7] + [b"A" * long_q] + qs[8:], rs[:7] + [b"A" * long_r] + rs[8:])
    bad.maxq, bad.maxr = 320, 480  # what the batched path can be told at most
    p = Path(300, 320, 480)
    try:
        want = orc.sw_batch(qs, rs, *sc, nthreads=8)
        assert p.call(how, good, sc) == 0
        check(good.results(), want)
        for _ in range(2):
            assert p.call(how, bad, sc) == 5  # SWIFT_ERR_CAPACITY
        good.score.zero()
        assert p.call(how, good, sc) == 0
        check(good.results(), want)
    finally:
        p.close()


@pytest.mark.parametrize("how", ["run", "enqueue"])
def test_longer_than_said_is_not_passed_over(orc, how):
    """A small call that said less than a pair's length and does not wait: it has
    no second path to take, and says so."""
    from swift_amd import align as A
    qs, rs = edge_pairs(random.Random(1), 200, 120, 200)
    b = A.PairBatch(qs, rs)
    p = Path(200, 320, 480)
    try:
        b.maxq, b.maxr = 90, 200
        assert p.call(how, b, (2, -1, -10, -1)) == 5
        b.maxq, b.maxr = 120, 200
        assert p.call(how, b, (2, -1, -10, -1)) == 0
        check(b.results(), orc.sw_batch(qs, rs, nthreads=8))
    finally:
        p.close()


def test_first_calls(orc):
    """The first call of a workspace, which makes its counters, on a stream that
    does not wait for the null stream: the screen and the kernel on its list."""
    qs, rs = edge_pairs(random.Random(3), 4100, 100, 160)
    want = orc.sw_batch(qs, rs, nthreads=8)
    from swift_amd import align as A
    b = A.PairBatch(qs, rs)
    for _ in range(6):
        p = Path()
        try:
            assert p.call("run", b, (2, -1, -10, -1), 0) == 0
            check(b.results(), want)
        finally:
            p.close()
