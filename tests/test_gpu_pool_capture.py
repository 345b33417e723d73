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
