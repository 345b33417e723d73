"""Freeing while a stream is being captured, by a thread that may, and while
kernels run on a stream that waits for nobody."""
import ctypes as C
import threading
import time

import pytest

pytestmark = pytest.mark.gpu
THREAD_LOCAL, RELAXED = 1, 2


@pytest.fixture(scope="module")
def hip():
    from swift_amd._lib import lib
    lib()
    return C.CDLL("libamdhip64.so")


def allocate(n):
    from swift_amd._lib import lib
    p = C.c_void_p()
    assert lib().swift_device_alloc(C.byref(p), n) == 0
    return p


@pytest.mark.parametrize("mode,own", [(THREAD_LOCAL, False), (RELAXED, False), (RELAXED, True)])
def test_free_beside_a_capture(hip, mode, own):
    from swift_amd._lib import lib
    from swift_amd.device import Stream
    p, s, got = allocate(1 << 20), Stream(), []
    assert hip.hipStreamBeginCapture(s.cptr, mode) == 0

    def work():
        got.append(lib().swift_device_free(p))
        q = allocate(1 << 20)
        got.append(lib().swift_device_free(q))

    if own:
        work()
    else:
        t = threading.Thread(target=work)
        t.start()
        t.join()
    graph = C.c_void_p()
    assert hip.hipStreamEndCapture(s.cptr, C.byref(graph)) == 0
    assert got == [0, 0]


@pytest.mark.parametrize("n", [1000, 1 << 20])
def test_free_waits_for_the_device(n):
    import torch
    from swift_amd._lib import lib
    p = allocate(n)
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(st):
        torch.cuda._sleep(100_000_000)  # some ten milliseconds
    done = st.record_event()
    t = time.perf_counter()
    assert lib().swift_device_free(p) == 0
    assert done.query(), time.perf_counter() - t


def test_first_batch_beside_a_capture(hip, orc):
    """A workspace's first call, on its own stream, while another thread's stream
    that the null stream waits for is being captured."""
    import random

    from swift_amd import align as A
    from test_gpu_sw_lean import check, edge_pairs
    from test_gpu_sw_status import Path
    qs, rs = edge_pairs(random.Random(9), 300, 100, 160)
    b, got = A.PairBatch(qs, rs), []
    s = C.c_void_p()
    assert hip.hipStreamCreate(C.byref(s)) == 0
    p = Path()
    assert hip.hipStreamBeginCapture(s, THREAD_LOCAL) == 0
    t = threading.Thread(target=lambda: got.append(p.call("run", b, (2, -1, -10, -1))))
    t.start()
    t.join()
    graph = C.c_void_p()
    end = hip.hipStreamEndCapture(s, C.byref(graph))
    p.close()
    assert got == [0] and end == 0
    assert hip.hipStreamDestroy(s) == 0
    check(b.results(), orc.sw_batch(qs, rs, nthreads=8))
