"""The plain path's route by lengths, pairs and the scratch its chunks may take
(a host function of libswift_amd.so: no GPU)."""
import ctypes as C

import pytest

GENERAL, PACKED, WAVE = range(3)
HELD = 1 << 24  # words of the no-allocation call's array
OWN = 1 << 30   # ... of the allocating call's


class Plan(C.Structure):  # PlainPlan, swift_amd/csrc/sw_host.hpp
    _fields_ = [(f, C.c_int) for f in ("route", "qlen", "rlen", "move_words", "form", "wave_rows",
                                       "packed_rows")] + [("wave_words", C.c_int64),
                                                          ("task_words", C.c_int64)]


# pairs, query and reference length, scratch
@pytest.mark.parametrize("n,ql,rl,words,route",
                         [(4095, 100, 300, OWN, WAVE), (4096, 100, 300, OWN, PACKED),
                          (4096, 320, 480, OWN, PACKED), (4096, 321, 480, OWN, WAVE),
                          (4200, 100, 300, HELD, PACKED), (20000, 128, 800, HELD, PACKED),
                          (4200, 256, 450, HELD, PACKED),
                          # past 16 rows a lane: by the chunk, not by the call
                          (4200, 257, 450, HELD, WAVE), (100000, 320, 480, HELD, WAVE),
                          (4200, 300, 200, HELD, WAVE), (4200, 300, 100, HELD, PACKED)])
def test_route(n, ql, rl, words, route):
    from swift_amd._lib import lib
    f = lib()._ZN5swift10plain_planERKNS_7ScoringEiiil
    f.restype = Plan
    f.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_int64]
    sc = (C.c_int * 4)(2, -1, -10, -1)
    assert f(sc, ql, rl, n, words).route == route
    lossless = (C.c_int * 4)(2, 0, -10, -1)
    assert f(lossless, ql, rl, n, words).route == GENERAL
