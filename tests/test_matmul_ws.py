"""lkhip_matmul's workspaces (lokal_amd/csrc/matmul_ws.h) on the CPU, over a
stand-in for the few HIP calls they make: a device of a given size that refuses
what does not fit, and keeps the last error until it is read, as HIP does."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
HIP = r"""
#pragma once
#include <cstddef>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
typedef struct FakeStream* hipStream_t;
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0, hipStreamCaptureStatusActive = 1 };
hipError_t hipGetDevice(int* d);
hipError_t hipSetDevice(int d);
hipError_t hipGetLastError();
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st);
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t s);
hipError_t hipFreeAsync(void* p, hipStream_t s);
hipError_t hipFree(void* p);
"""
PROBE = r"""
#include <chrono>
#include <future>
#include <map>
#include <mutex>
#include <cstdint>
#include "matmul_ws.h"
static std::mutex mu;
static std::map<void*, size_t> live;
static size_t room_left, device_waits, recorded;
static hipError_t last;
static uintptr_t next_ptr = 4096;
static hipStream_t capturing;
static void* graphs;  // the last allocation made under capture, freed there too
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { std::lock_guard<std::mutex> l(mu); const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    *st = s && s == capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t s) {
    std::lock_guard<std::mutex> l(mu);
    if (n > room_left) return last = hipErrorOutOfMemory;
    room_left -= n;
    *p = (void*)(next_ptr += 4096);
    live[*p] = n;
    if (s && s == capturing) graphs = *p;
    return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t s) {
    std::lock_guard<std::mutex> l(mu);
    if (s && s == capturing && p != graphs) { recorded++; return hipSuccess; }  // a node of the graph
    room_left += live.at(p);
    live.erase(p);
    return hipSuccess;
}
hipError_t hipFree(void* p) { device_waits++; return hipFreeAsync(p, nullptr); }

static lkws::Pool* pool;
extern "C" {
void start(size_t bytes) { delete pool; pool = new lkws::Pool; live.clear(); room_left = bytes; last = hipSuccess; capturing = nullptr; device_waits = recorded = 0; }
// one call with a workspace of n bytes: whether it had one, and the bytes allocated while it ran
int call(hipStream_t s, size_t n, size_t* held) {
    lkws::Scratch ws(*pool, s);
    void* p = ws.get(n);
    size_t sum = 0;
    for (auto& kv : live) sum += kv.second;
    *held = sum;
    return p != nullptr;
}
// whether a call on t from another thread is through (1) or waits (0) while one on s holds its workspace
int beside(hipStream_t s, hipStream_t t) {
    std::future<int> f;
    bool through;
    {
        lkws::Scratch ws(*pool, s);
        ws.get(1 << 20);
        f = std::async(std::launch::async, [t] { size_t held; return call(t, 1 << 20, &held); });
        through = f.wait_for(std::chrono::milliseconds(s == t ? 100 : 5000)) == std::future_status::ready;
    }
    return f.get() && through;
}
size_t waits() { return device_waits; }
size_t frees_recorded() { return recorded; }
void capture(hipStream_t s) { capturing = s; }
int last_error() { return (int)hipGetLastError(); }
size_t held() { size_t sum = 0; for (auto& kv : live) sum += kv.second; return sum; }
void made(hipStream_t s) { lkws::stream_created(*pool, s); }
void ended(hipStream_t s) { lkws::stream_destroyed(*pool, s); }
void weight(int made) { made ? lkws::weight_created(*pool) : lkws::weight_destroyed(*pool); }
}
"""
MB = 1 << 20


@pytest.fixture(scope="module")
def ws(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("ws")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime_api.h").write_text(HIP)
    (d / "probe.cpp").write_text(PROBE)
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-pthread", "-I", str(d), "-I",
                    str(ROOT / "lokal_amd" / "csrc"), str(d / "probe.cpp"), "-o", str(d / "probe.so")], check=True)
    lib = C.CDLL(str(d / "probe.so"))
    lib.start.argtypes = [C.c_size_t]
    lib.call.argtypes = [C.c_void_p, C.c_size_t, C.c_void_p]
    lib.held.restype = lib.waits.restype = lib.frees_recorded.restype = C.c_size_t
    lib.made.argtypes = lib.ended.argtypes = lib.capture.argtypes = [C.c_void_p]
    lib.beside.argtypes = [C.c_void_p, C.c_void_p]

    def call(stream, n):
        held = C.c_size_t()
        return lib.call(stream, n, C.byref(held)), held.value

    lib.run = call
    return lib


def test_growth_that_does_not_fit(ws):
    """A kept buffer asks for twice its size to grow; where that does not fit, the
    call still gets what it needs, and no error is left for the launch checks."""
    ws.start(10 * MB)
    assert ws.run(None, 3 * MB) == (1, 4 * MB)
    assert ws.run(None, 5 * MB)[0] == 1  # 8 MB beside the 4 do not fit
    assert ws.last_error() == 0 and ws.held() == 5 * MB
    assert ws.run(None, 10 * MB)[0] == 1  # nor 10 beside the 5
    assert ws.last_error() == 0 and ws.held() == 10 * MB


@pytest.mark.parametrize("stream", [None, 1, 2])
def test_no_memory_leaves_no_error(ws, stream):
    """A workspace larger than the device, on a kept stream (None, 1) or another."""
    ws.start(6 * MB)
    ws.made(1)
    assert ws.run(stream, MB)[0] == 1
    assert ws.run(stream, 7 * MB)[0] == 0
    assert ws.last_error() == 0
    assert ws.run(stream, 6 * MB)[0] == 1  # nothing is held on to
    assert ws.last_error() == 0


def test_streams_do_not_wait_for_each_other(ws):
    """A call holds its own stream's buffer only: calls on one stream share it in
    turn, calls on two streams go on beside each other."""
    ws.start(100 * MB)
    ws.made(1), ws.made(2)
    assert ws.beside(1, 2) == 1 and ws.beside(None, 1) == 1
    assert ws.beside(1, 1) == 0 and ws.beside(None, None) == 0
    assert ws.held() == 3 * 4 * MB


def test_buffers_are_bounded_and_given_back(ws):
    """At most 16 buffers, none above 64 MB, none for a stream that was not made
    here or is being captured; a destroyed stream's and, with the last weight,
    all of them are freed without waiting for the device."""
    ws.start(1 << 40)
    ws.weight(1), ws.weight(1)
    for s in range(1, 20):
        ws.made(s)
        assert ws.run(s, 64 * MB)[0] == 1
    assert ws.held() == 16 * 64 * MB
    assert ws.run(1, 64 * MB + 1) == (1, 17 * 64 * MB + 1) and ws.held() == 16 * 64 * MB
    assert ws.run(99, MB) == (1, 16 * 64 * MB + MB) and ws.held() == 16 * 64 * MB
    ws.ended(3)
    assert ws.held() == 15 * 64 * MB
    ws.capture(19)
    assert ws.run(19, MB) == (1, 15 * 64 * MB + MB) and ws.held() == 15 * 64 * MB
    ws.capture(None)
    assert ws.run(19, MB)[0] == 1 and ws.held() == 15 * 64 * MB + 4 * MB
    ws.weight(0)
    assert ws.held() == 15 * 64 * MB + 4 * MB
    ws.weight(0)
    assert ws.held() == 0 and ws.waits() == 0
    ws.weight(1)
    assert ws.run(5, MB)[0] == 1 and ws.held() == 4 * MB


def test_no_free_is_recorded_into_a_capture(ws):
    """The last weight goes while a stream with a kept buffer is being captured: the
    free would become a node of that graph, so the buffer stays and is used and freed
    later; the other streams' go.  A destroyed stream's goes in any case."""
    ws.start(100 * MB)
    ws.weight(1)
    ws.made(1), ws.made(2)
    assert ws.run(1, MB)[0] == 1 and ws.run(2, MB)[0] == 1
    ws.capture(1)
    ws.weight(0)
    assert ws.frees_recorded() == 0 and ws.held() == 4 * MB
    ws.capture(None)
    ws.weight(1)
    assert ws.run(1, MB) == (1, 4 * MB)
    ws.weight(0)
    assert ws.held() == 0
    ws.weight(1)
    assert ws.run(2, MB)[0] == 1
    ws.capture(2)
    ws.ended(2)
    assert ws.frees_recorded() == 0 and ws.held() == 0
