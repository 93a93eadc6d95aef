"""The results' way to the host (csrc/host_copy.hip) on the CPU: its source compiled against a stand-in for the HIP runtime
whose copies are queued and done when something waits for them, so that bytes taken before they arrived are wrong ones.

Every row's bytes, rows that were not asked for untouched, rows with gaps waited for together, memory that HIP allocated
(page-locked, device) written by the device itself, and a model without page-locked chunks still served.
"""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#pragma once
#include <stddef.h>
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
typedef struct stream_t* hipStream_t;
typedef struct event_t* hipEvent_t;
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum { hipEventDisableTiming = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost, hipMemoryTypeDevice };
struct hipPointerAttribute_t { int type; };
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags);
hipError_t hipHostFree(void* p);
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags);
hipError_t hipEventDestroy(hipEvent_t e);
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s);
hipError_t hipEventSynchronize(hipEvent_t e);
hipError_t hipStreamSynchronize(hipStream_t s);
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t s);
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p);
hipError_t hipGetLastError();
"""

HARNESS = r"""
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <string.h>
#include <deque>
#include <vector>
#include "host_copy.h"
struct event_t { size_t at; };
struct op { char* dst; const char* src; size_t n; };
static std::deque<op> queue;
static size_t done, issued;
static int waits, direct, no_memory, fail_at;
static std::vector<std::pair<const char*, size_t>> own, pinned;
static bool in(const std::vector<std::pair<const char*, size_t>>& v, const void* p) {
    for (auto& r : v) if ((const char*)p >= r.first && (const char*)p < r.first + r.second) return true;
    return false;
}
static void until(size_t at) {
    for (; done < at; done++) { memcpy(queue.front().dst, queue.front().src, queue.front().n); queue.pop_front(); }
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (no_memory) return hipErrorOutOfMemory;
    *p = malloc(n); own.push_back({(char*)*p, n}); return hipSuccess;
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = new event_t(); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { e->at = issued; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { waits++; until(e->at); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { waits++; until(issued); return hipSuccess; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
    if (fail_at && !--fail_at) return hipErrorInvalidValue;
    queue.push_back({(char*)dst, (const char*)src, n}); issued++;
    direct += !in(own, dst);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    a->type = in(own, p) || in(pinned, p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
extern "C" {
void* make(int without) { no_memory = without; own.clear(); pinned.clear(); return host_copy_create(); }
void unmake(void* c) { host_copy_destroy((host_copy*)c); }
void pin(const char* p, size_t n) { pinned.push_back({p, n}); }
int rows(void* c, const void* dev, size_t bytes, size_t n, void* const* dst, int fail, int* waited, int* straight, int* left) {
    waits = direct = 0; fail_at = fail;
    const int e = host_copy_rows((host_copy*)c, nullptr, dev, bytes, n, dst);
    *waited = waits; *straight = direct; *left = (int)(issued - done);
    until(issued); fail_at = 0;
    return e;
}
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_copy")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (d / "harness.cpp").write_text(HARNESS)
    csrc = os.path.join(ROOT, "vitna-anchor_amd", "csrc")
    out = str(d / "libharness.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fPIC", "-shared", "-pthread", "-I", str(d), "-I", csrc, "-o", out, str(d / "harness.cpp"),
                    "-x", "c++", os.path.join(csrc, "host_copy.hip")], check=True)
    L = C.CDLL(out)
    L.make.restype = C.c_void_p
    L.unmake.argtypes = [C.c_void_p]
    L.pin.argtypes = [C.c_void_p, C.c_size_t]
    L.rows.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_size_t, C.c_void_p, C.c_int] + [C.POINTER(C.c_int)] * 3
    return L


class Rows:
    """n rows of `bytes` bytes on the device and places for them, those of `want` asked for; stride between the places."""

    def __init__(self, n, bytes_, want, stride=None, seed=1):
        self.n, self.bytes, self.want = n, bytes_, sorted(want)
        self.dev = np.random.RandomState(seed).randint(0, 256, (n, bytes_), dtype=np.uint8)
        self.out = np.full((n, stride or bytes_), 7, np.uint8)
        self.dst = np.zeros(n, np.uintp)
        self.dst[self.want] = self.out.ctypes.data + np.array(self.want, np.uintp) * np.uintp(self.out.strides[0])

    def run(self, lib, c, fail=0):
        w, s, left = C.c_int(), C.c_int(), C.c_int()
        rc = lib.rows(c, self.dev.ctypes.data, self.bytes, self.n, self.dst.ctypes.data, fail, C.byref(w), C.byref(s), C.byref(left))
        if rc == 0:
            assert left.value == 0, "copies under way at the return"
            for i in range(self.n):
                assert np.array_equal(self.out[i, :self.bytes], self.dev[i]) if i in self.want else (self.out[i] == 7).all(), i
            assert (self.out[:, self.bytes:] == 7).all()
        return rc, w.value, s.value


@pytest.fixture(params=[0, 1], ids=["chunks", "no chunks"])
def copier(lib, request):
    c = lib.make(request.param)
    assert bool(c) != bool(request.param)
    yield lib, c
    lib.unmake(c)


@pytest.mark.parametrize("n,bytes_", [(1, 1), (1, 4000), (1, 65536), (1, 65540), (1, 607744), (2, 1 << 20), (1, (1 << 21) - 4), (1, 1 << 21),
                                      (5, 524288), (33, 131084), (40, 607744), (700, 4000), (1024, 16)])
def test_bytes(copier, n, bytes_):
    lib, c = copier
    for want in (range(n), [0], [n - 1], range(0, n, 2), range(n // 3, n), []):
        for stride in (None, bytes_ + 64):
            assert Rows(n, bytes_, want, stride).run(lib, c)[0] == 0


def test_gaps_are_waited_for_once(lib):
    """Small rows with gaps: one wait, nothing copied past the chunks; more runs than are held, or than 16 MB hold, a wait
    for each lot."""
    c = lib.make(0)
    assert Rows(200, 4000, range(0, 200, 2)).run(lib, c) == (0, 1, 0)
    assert Rows(64, 4000, [0, 1, 5, 6, 7, 60]).run(lib, c) == (0, 1, 0)
    assert Rows(1024, 400, range(0, 1024, 2)).run(lib, c) == (0, 1, 0)
    assert Rows(2048, 400, range(0, 2048, 2)).run(lib, c) == (0, 2, 0)
    assert Rows(1024, 65536, range(0, 1024, 2)).run(lib, c) == (0, 2, 0)
    lib.unmake(c)


def test_memory_of_hip_is_written_directly(lib):
    """Rows in page-locked (or device) memory: a copy each and one wait; mixed with rows in ordinary memory, each its way."""
    for n, b, pinned, straight in ((1, 4000, range(1), 1), (8, 160000, range(8), 8), (32, 607744, range(32), 32), (200, 4000, range(200), 200),
                                   (40, 607744, range(10, 15), 5), (40, 131072, range(10, 15), 5 + 10), (200, 4000, range(40, 80), None)):
        c = lib.make(0)
        r = Rows(n, b, range(n))
        lib.pin(r.out[pinned[0]:].ctypes.data, len(pinned) * b)
        rc, waits, direct = r.run(lib, c)
        assert rc == 0
        if len(pinned) == n:
            assert waits == 1
        assert straight is None or direct == straight
        lib.unmake(c)


@pytest.mark.parametrize("fail", [1, 2, 5, 30])
def test_a_failing_copy(lib, fail):
    """A copy that cannot be issued: the error, with nothing on its way to the chunks, which the next call uses."""
    c = lib.make(0)
    for n, b, want in ((200, 4000, range(0, 200, 2)), (60, 607744, range(60)), (6, 160000, range(6))):
        r = Rows(n, b, want)
        rc, _, _ = r.run(lib, c, fail)
        assert rc == (1 if fail <= {200: 100, 60: 70, 6: 6}[n] else 0)
        assert Rows(n, b, want, seed=9).run(lib, c)[0] == 0
    lib.unmake(c)
