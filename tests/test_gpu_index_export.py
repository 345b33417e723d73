"""The index's arrays read back: one alone or all, over more hashes than go at
once, and in the time that copies of as many bytes take."""
import ctypes as C
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def least(f, reps=5):
    best = 1e9
    for _ in range(reps):
        t = time.perf_counter()
        f()
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("k,thr", [(1, 1 << 30), (5, 40), (12, 2)])
def test_arrays(orc, k, thr):
    from swift_amd import search, synth
    from swift_amd._lib import check, lib
    rng = np.random.default_rng(k)
    seqs = [synth.random_bases(rng, n).tobytes() for n in (70_000, 11)]
    ix = search.Index.from_sequences(seqs, k, thr)
    want = orc.Index(seqs, k, thr).arrays()
    got = ix.arrays()
    for f in ("start", "count", "actual"):
        assert np.array_equal(got[f], want[f]), f
        one = np.full(4 ** k, -7, np.int32)
        args = [one.ctypes.data_as(C.POINTER(C.c_int32)) if g == f else None
                for g in ("start", "count", "actual")]
        check(lib().swift_index_export(ix._h, *args, None, None))
        assert np.array_equal(one, want[f]), f
    ix.close()


def test_time():
    """1.7 times the copies' with loops over the hashes on the host, 1.02 without."""
    from swift_amd import search, synth
    from swift_amd.device import DeviceBuffer
    ix = search.Index.from_sequences([synth.random_bases(np.random.default_rng(1), 9000).tobytes()],
                                     12, 1000)
    b = DeviceBuffer(4 << 24)
    copies = least(lambda: [b.download(np.int32, 1 << 24) for _ in range(3)])
    took = least(ix.arrays)
    ix.close()
    assert took < 1.35 * copies, (took, copies)
