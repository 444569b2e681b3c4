"""The lanes of large copies (mkde_copy.cpp) on the CPU, against a stand-in for the
HIP runtime whose streams copy when an event or a stream is waited for: bytes of every
size class in both directions, every device of a process with lanes of its own, several
threads at once, failures of every call, and nothing left after the lanes are given
back."""
import os
import shutil
import subprocess

import pytest

import mgpukde_tiled_amd as M

CSRC = os.path.join(os.path.dirname(M.__file__), "csrc")

HIP = r"""
#pragma once
#include <stddef.h>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum { hipStreamNonBlocking = 1, hipEventDisableTiming = 2, hipHostMallocDefault = 0 };
struct Stream;
struct Event;
typedef Stream *hipStream_t;
typedef Event *hipEvent_t;
hipError_t hipSetDevice(int);
hipError_t hipGetLastError();
hipError_t hipStreamCreateWithFlags(hipStream_t *, unsigned);
hipError_t hipStreamDestroy(hipStream_t);
hipError_t hipStreamSynchronize(hipStream_t);
hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned);
hipError_t hipEventDestroy(hipEvent_t);
hipError_t hipEventRecord(hipEvent_t, hipStream_t);
hipError_t hipEventSynchronize(hipEvent_t);
hipError_t hipHostMalloc(void **, size_t, unsigned);
hipError_t hipHostFree(void *);
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t);
"""

MAIN = r"""
#include "mkde_copy.h"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

// queued work runs when something waits for it
struct Stream { int device; std::mutex mu; std::deque<std::function<void()>> q; };
struct Event { int device; Stream *s = nullptr; std::atomic<bool> done{true}; };
static thread_local int cur = 0;
static std::atomic<int> live_streams[4], live_events, live_pinned, fail_at{-1}, calls;
static std::atomic<long> wrong_device;
static hipError_t step(hipError_t e) { return fail_at >= 0 && calls++ == fail_at ? e : hipSuccess; }
static void run(Stream *s, Event *until)
{
    std::lock_guard<std::mutex> lk(s->mu);
    while (!s->q.empty() && !(until && until->done)) { auto f = s->q.front(); s->q.pop_front(); f(); }
}
hipError_t hipSetDevice(int d) { cur = d; return step(hipErrorUnknown); }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    if (hipError_t e = step(hipErrorOutOfMemory)) return e;
    *s = new Stream{cur}; ++live_streams[cur]; return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { run(s, nullptr); --live_streams[s->device]; delete s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { run(s, nullptr); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    if (hipError_t r = step(hipErrorOutOfMemory)) return r;
    *e = new Event{cur}; ++live_events; return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { --live_events; delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    if (hipError_t r = step(hipErrorUnknown)) return r;
    if (e->device != s->device) ++wrong_device;
    e->s = s; e->done = false;
    std::lock_guard<std::mutex> lk(s->mu);
    s->q.push_back([e] { e->done = true; });
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { if (!e->done) run(e->s, e); return step(hipErrorUnknown); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (hipError_t r = step(hipErrorOutOfMemory)) return r;
    *p = malloc(n); ++live_pinned; return hipSuccess;
}
hipError_t hipHostFree(void *p) { free(p); --live_pinned; return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st)
{
    if (hipError_t r = step(hipErrorUnknown)) return r;
    if (st->device != cur) ++wrong_device;
    std::lock_guard<std::mutex> lk(st->mu);
    st->q.push_back([=] { memcpy(d, s, n); });
    return hipSuccess;
}

#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); exit(1); } } while (0)

static std::vector<unsigned char> bytes(size_t n, unsigned seed)
{
    std::vector<unsigned char> v(n);
    for (size_t i = 0; i < n; ++i) v[i] = (unsigned char)((i * 2654435761u + seed) >> 13);
    return v;
}
// 1: with lanes, 0: not one for lanes, -1: error
static int copy(int dev, hipStream_t shared, size_t n, bool to_host, unsigned seed)
{
    std::vector<unsigned char> a = bytes(n, seed), b(n);
    bool done = false;
    cur = dev;   // the caller's part
    const hipError_t e = mkde_copy::run(dev, shared, b.data(), a.data(), n, to_host, &done);
    if (e != hipSuccess) return -1;
    if (done) CHECK(a == b);
    return done;
}

int main()
{
    using namespace mkde_copy;
    const size_t MB = (size_t)1 << 20;
    // small copies are none for lanes, and few large ones do not earn them
    CHECK(copy(0, nullptr, MIN_TO_HOST - 1, true, 1) == 0 && copy(0, nullptr, MIN_TO_DEVICE - 1, false, 1) == 0);
    CHECK(copy(0, nullptr, MIN_MOVED / 2, true, 2) == 0 && live_pinned == 0);
    // every device gets lanes of its own, as many as the first
    for (int dev = 0; dev < 4; ++dev) {
        CHECK(copy(dev, nullptr, MIN_MOVED, true, dev) == 1);
        CHECK(live_streams[dev] == 8);
        for (size_t n : {MIN_TO_HOST, 2 * MB - 1, 2 * MB, 2 * MB + 1, 9 * MB + 77, 17 * MB + 5})
            CHECK(copy(dev, nullptr, n, true, (unsigned)n) == 1);
        for (size_t n : {MIN_TO_DEVICE, MIN_TO_DEVICE + 1, MIN_TO_DEVICE + 3 * MB - 3}) CHECK(copy(dev, nullptr, n, false, (unsigned)n) == 1);
    }
    // on the caller's stream; below its own limit not at all
    Stream *own = new Stream{1};
    CHECK(copy(1, own, MIN_SHARED - 1, true, 3) == 0);
    CHECK(copy(1, own, MIN_SHARED + 9, true, 3) == 1 && copy(1, own, MIN_SHARED + 9, false, 4) == 1);
    // a device number beyond the table is none for lanes
    CHECK(copy(64, nullptr, MIN_MOVED, true, 1) == 0 && copy(-1, nullptr, MIN_MOVED, true, 1) == 0);
    // more copies than lanes, on one device and on two
    std::vector<std::thread> th;
    std::atomic<int> ok{0};
    for (int i = 0; i < 6; ++i) th.emplace_back([&, i] { for (int k = 0; k < 4; ++k) ok += copy(i % 2, nullptr, (3 + 5 * i + k) * MB + i, k % 2, i) >= 0; });
    for (std::thread &t : th) t.join();
    CHECK(ok == 24 && live_streams[0] <= 12 && live_streams[1] <= 12 && wrong_device == 0);
    // nothing is left
    for (int dev = 0; dev < 4; ++dev) give_back(dev);
    CHECK(live_pinned == 0 && live_events == 0);
    for (int dev = 0; dev < 4; ++dev) CHECK(live_streams[dev] == 0);
    give_back(0);
    give_back(64);
    // a call that fails, each in turn: the copy is right, or none, or says so; the next is right
    int failed = 0, none = 0, right = 0;
    for (int at = 0; at < 150; ++at) {
        calls = 0;
        fail_at = at;
        const int r = copy(2, nullptr, MIN_TO_DEVICE + 3, at % 2, at);
        fail_at = -1;
        (r < 0 ? failed : r ? right : none)++;
        CHECK(copy(2, nullptr, MIN_TO_DEVICE + 3, at % 2, at) == 1);
        if (at % 7 == 0) give_back(2);
    }
    CHECK(failed > 20 && right > 10);
    give_back(2);
    CHECK(live_pinned == 0 && live_events == 0 && live_streams[2] == 0);
    // no pinned memory at all
    th.clear();
    for (int at = 0; at < 3; ++at) {
        calls = 0;
        fail_at = at;   // the first lane's first calls; the others are not tried then
        CHECK(copy(3, nullptr, 2 * MB, true, 1) == 0 || at == 2);
        fail_at = -1;
    }
    delete own;
    printf("ok\n");
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_lanes(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "lanes")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-I", str(tmp_path), "-I", CSRC, str(tmp_path / "main.cpp"),
                    os.path.join(CSRC, "mkde_copy.cpp"), "-o", exe, "-pthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
