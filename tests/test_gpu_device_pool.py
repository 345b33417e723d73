"""Device memory kept between owners, and uploads of many sizes."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# below and past the sizes the runtime stages in one piece
@pytest.mark.parametrize("n", [1, (4 << 20) - 1, 4 << 20, (5 << 20) + 1, (33 << 20) + 12345])
def test_upload_round_trip(n):
    from swift_amd.device import DeviceBuffer
    a = np.random.default_rng(n).integers(0, 256, n, dtype=np.uint8)
    b = DeviceBuffer.from_array(a)
    assert np.array_equal(b.download(np.uint8, n), a)


def test_blocks_are_not_shared():
    """Threads that allocate, fill, read back and free sizes of few classes, at
    once: nobody sees another's bytes; unknown and null pointers are refused
    and accepted as before."""
    from swift_amd._lib import lib
    from swift_amd.device import DeviceBuffer
    bad = []

    def work(t):
        rng = np.random.default_rng(t)
        held = []
        for i in range(60):
            n = int(rng.choice((100, 4096, 70_000, 5 << 20))) + int(rng.integers(0, 200))
            b = DeviceBuffer(n)
            v = (t * 60 + i) % 251
            b.upload(np.full(n, v, np.uint8))
            held.append((b, n, v))
            if len(held) > 4:
                b, n, v = held.pop(int(rng.integers(0, len(held))))
                if not (b.download(np.uint8, n) == v).all():
                    bad.append((t, i, n))
                b.free()
        for b, n, v in held:
            if not (b.download(np.uint8, n) == v).all():
                bad.append((t, n))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(6)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad
    assert lib().swift_device_free(None) == 0
    p = C.c_void_p()
    assert lib().swift_device_alloc(C.byref(p), 1 << 50) != 0


def test_index_after_index():
    """Indexes built one after another in the same blocks give the same hits."""
    from swift_amd import search, synth
    rng = np.random.default_rng(1)
    for size in (300_000, 40_000, 300_001):
        seqs = [synth.random_bases(rng, size).tobytes()]
        reads, _ = synth.sample_reads(rng, [np.frombuffer(seqs[0], np.uint8)], 50, 100, 0.01, 0.0)
        got = []
        for _ in range(2):
            ix = search.Index.from_sequences(seqs, 12, 1000)
            r = ix.align_reads(reads, 3)
            got.append((r.cols, r.qry_cons))
            ix.close()
        for f in got[0][0]:
            assert np.array_equal(got[0][0][f], got[1][0][f]), f
        assert got[0][1] == got[1][1]
