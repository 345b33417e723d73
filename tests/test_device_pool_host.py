"""The pool of freed device memory (swift_amd/csrc/device_pool.cpp) on the CPU,
over a HIP whose device memory is a table of addresses: what it hands out is
mapped and has one owner, whatever is freed twice, elsewhere or too late."""
import ctypes as C
import os
import subprocess
import threading

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "swift_amd", "csrc")

HIP = r"""
#pragma once
#include <cstddef>
#define __host__
#define __device__
#define __forceinline__ inline
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
typedef void *hipDeviceptr_t;
typedef void *hipStream_t;
hipError_t hipMalloc(void **p, size_t n);
hipError_t hipFree(void *p);
hipError_t hipGetDevice(int *d);
hipError_t hipDeviceSynchronize();
hipError_t hipGetLastError();
hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *size, hipDeviceptr_t p);
const char *hipGetErrorString(hipError_t e);
"""

MEMORY = r"""
#include <map>
#include <mutex>
#include "device_pool.hpp"
static std::recursive_mutex mu;
static std::map<char *, size_t> mapped;
static size_t in_use, limit = ~(size_t)0;
static int waits, device, last, refuse;  // frees to refuse, as in a capture
static void (*on_sync)();
static void wait() {
    ++waits;
    if (on_sync) { auto f = on_sync; on_sync = nullptr; f(); }
}
hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (n > limit - in_use) return last = hipErrorOutOfMemory;
    char *at = (char *)0x100000;  // the lowest gap
    for (auto &m : mapped) {
        if (m.first >= at + n) break;
        at = m.first + m.second;
    }
    mapped[at] = n;
    in_use += n;
    *p = at;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    wait();
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (refuse > 0) {
        --refuse;
        return last = hipErrorInvalidValue;
    }
    auto it = mapped.find((char *)p);
    if (it == mapped.end()) return last = hipErrorInvalidValue;
    in_use -= it->second;
    mapped.erase(it);
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) { *d = device; return hipSuccess; }
hipError_t hipDeviceSynchronize() { wait(); return hipSuccess; }
hipError_t hipGetLastError() { int e = last; last = 0; return e; }
hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *size, hipDeviceptr_t p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    auto it = mapped.upper_bound((char *)p);
    if (it == mapped.begin()) return last = hipErrorInvalidValue;
    --it;
    if ((char *)p >= it->first + it->second) return last = hipErrorInvalidValue;
    *base = it->first;
    *size = it->second;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return ""; }
extern "C" {
int t_alloc(void **p, size_t n) { return swift::pool_alloc(p, n, false); }
int t_array(void **p, size_t n) { return swift::pool_alloc(p, n, true); }
int t_release(void *p) { return swift::pool_free(p, false); }
int t_waits() { return waits; }
void t_refuse(int n) { refuse = n; }
int t_free(void *p) { return swift::pool_free(p, true); }
int t_device_malloc(void **p, size_t n) { return swift::device_malloc(p, n); }
int t_trim() { return swift::pool_trim(); }
int t_hip_malloc(void **p, size_t n) { return hipMalloc(p, n); }
int t_hip_free(void *p) { return hipFree(p); }
void t_limit(size_t n) { limit = n; }
void t_device(int d) { device = d; }
void t_on_sync(void (*f)()) { on_sync = f; }
size_t t_mapped(void *p) {  // bytes mapped from p on, p the start of its block
    auto it = mapped.find((char *)p);
    return it == mapped.end() ? 0 : it->second;
}
}
"""

SYNC = C.CFUNCTYPE(None)


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "memory.cpp").write_text(MEMORY)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", f"-I{d}", f"-I{CSRC}", "-o",
                    str(d / "pool.so"), str(d / "memory.cpp"),
                    os.path.join(CSRC, "device_pool.cpp")], check=True)
    return d


class Pool:
    def __init__(self, so):
        self.lib = C.CDLL(str(so))
        for f in ("alloc", "array", "hip_malloc", "device_malloc"):
            getattr(self.lib, "t_" + f).argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        for f in ("free", "release", "hip_free", "mapped"):
            getattr(self.lib, "t_" + f).argtypes = [C.c_void_p]
        self.lib.t_limit.argtypes = [C.c_size_t]
        self.lib.t_mapped.restype = C.c_size_t

    def alloc(self, n, how="alloc"):
        p = C.c_void_p()
        rc = getattr(self.lib, "t_" + how)(C.byref(p), n)
        return p.value if rc == 0 else None

    def __getattr__(self, name):
        return getattr(self.lib, "t_" + name)


@pytest.fixture
def pool(library, tmp_path):
    so = tmp_path / "pool.so"  # a library of its own: an empty pool
    so.write_bytes((library / "pool.so").read_bytes())
    return Pool(so)


def test_kept_blocks_are_used_again(pool):
    a = pool.alloc(1000)
    assert pool.free(a) == 0 and pool.mapped(a) >= 1000
    assert pool.alloc(1010) == a


def test_second_free_is_refused(pool):
    """... and unmaps nothing that the next owner is handed."""
    a = pool.alloc(1000)
    assert pool.free(a) == 0
    assert pool.free(a) != 0
    b = pool.alloc(1000)
    assert b is not None and pool.mapped(b) >= 1000
    assert pool.alloc(1000) != b


def test_second_free_during_the_first(pool):
    """The second comes while the first waits for the device."""
    a = pool.alloc(1000)
    got = []
    again = SYNC(lambda: got.append(pool.free(a)))
    pool.on_sync(again)
    assert pool.free(a) == 0 and got and got[0] != 0
    b = pool.alloc(1000)
    assert pool.mapped(b) >= 1000 and pool.alloc(1000) != b


def test_kept_memory_is_given_back(pool):
    """To the library's own allocations, in the pool or beside it, before one
    fails; to others by a trim, on the current device only."""
    size = 1 << 20
    pool.limit(4 * size + 4096)
    blocks = [pool.alloc(size) for _ in range(4)]
    for how in ("alloc", "device_malloc"):
        for b in blocks:
            assert pool.free(b) == 0
        p = pool.alloc(3 * size, how)
        assert p is not None
        assert pool.alloc(2 * size, how) is None
        assert pool.free(p) == 0 if how == "alloc" else pool.hip_free(p) == 0
        blocks = [pool.alloc(size) for _ in range(4)]
        assert None not in blocks
    pool.device(1)
    assert pool.alloc(size) is None  # no room: this device keeps nothing
    pool.device(0)
    for b in blocks:
        assert pool.free(b) == 0
    pool.device(1)
    assert pool.trim() == 0 and pool.alloc(size, "hip_malloc") is None
    pool.device(0)
    assert pool.trim() == 0 and pool.alloc(4 * size, "hip_malloc") is not None


def test_pointers_given_to_hip_free(pool):
    """A block the caller unmapped itself: a smaller allocation at its address
    is not kept under the old size, and what is unmapped is not handed out."""
    a = pool.alloc(100_000)
    assert pool.hip_free(a) == 0
    assert pool.free(a) != 0  # as hipFree answers
    a = pool.alloc(100_000)
    assert pool.hip_free(a) == 0
    b = pool.alloc(1000, "hip_malloc")
    assert b == a and pool.free(b) == 0
    c = pool.alloc(100_000)
    assert pool.mapped(c) >= 100_000
    # freed here and there
    assert pool.free(c) == 0 and pool.hip_free(c) == 0
    d = pool.alloc(1000, "hip_malloc")
    assert d == c
    e = pool.alloc(100_000)
    assert e != d and pool.mapped(e) >= 100_000
    assert pool.trim() == 0 and pool.mapped(d) == 1000


def test_others_allocate_while_blocks_are_given_back(pool):
    """hipFree waits for the device: the pool's lock is not held meanwhile."""
    assert pool.free(pool.alloc(1000)) == 0
    got = []

    def from_another_thread():
        t = threading.Thread(target=lambda: got.append(pool.alloc(5000)))
        t.start()
        t.join(5)
        got.append(t.is_alive())

    again = SYNC(from_another_thread)
    pool.on_sync(again)
    assert pool.trim() == 0
    assert got[0] is not False and got[-1] is False, got


def test_a_refused_free_loses_nothing(pool):
    """A block that hipFree refuses, in a thread that captures a stream, stays."""
    a = pool.alloc(1000)
    assert pool.free(a) == 0
    pool.refuse(1)
    assert pool.trim() == 0 and pool.mapped(a) >= 1000
    assert pool.alloc(1000) == a
    assert pool.free(a) == 0 and pool.trim() == 0 and pool.mapped(a) == 0


def test_the_oldest_go_first(pool):
    """1 GiB at most is kept: four blocks of 208 MiB, as 200 are rounded up to."""
    size = 200 << 20
    blocks = [pool.alloc(size) for _ in range(7)]
    for b in blocks:
        assert pool.free(b) == 0
    kept = [pool.mapped(b) > 0 for b in blocks]
    assert kept == [False] * 3 + [True] * 4


def test_a_block_let_go_unwaited(pool):
    """... is nobody's until the device has been waited for: by an allocation that
    may, once for all that went before, or by a free."""
    a, b = pool.alloc(1000), pool.alloc(1000)
    c, d = pool.alloc(9000), pool.alloc(9000)
    for p in (a, b, c):
        assert pool.release(p) == 0
    assert pool.alloc(1000) not in (a, b) and pool.waits() == 0
    assert pool.alloc(1000, "array") == b and pool.waits() == 1
    assert pool.alloc(1000, "array") == a and pool.alloc(9000) == c and pool.waits() == 1
    # one that goes during the wait is not covered by it
    late = SYNC(lambda: pool.release(d))
    assert pool.release(a) == 0
    pool.on_sync(late)
    assert pool.alloc(1000, "array") == a and pool.waits() == 2
    assert pool.alloc(9000) != d
    # a free's wait covers what was let go before
    assert pool.release(b) == 0 and pool.free(a) == 0 and pool.waits() == 3
    assert pool.alloc(1000) == a and pool.alloc(1000) == b and pool.alloc(9000) == d
    # a refused wait: new memory
    assert pool.release(b) == 0
    pool.refuse(1)
    assert pool.alloc(1000, "array") not in (None, b)
    # a second free of it, and giving it back
    assert pool.free(b) != 0 and pool.release(b) != 0
    assert pool.trim() == 0 and pool.mapped(b) == 0


def test_workspaces_ask_the_pool():
    """No allocation of device memory in the library goes past the pool."""
    for f in sorted(os.listdir(CSRC)):
        text = open(os.path.join(CSRC, f)).read()
        if not f.startswith("device_pool"):
            assert "hipMalloc(" not in text, f
