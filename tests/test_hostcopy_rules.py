"""Which way the copies of the host-pointer entry points take (csrc/zq3d_hostcopy.h), compiled with g++ against a
HIP runtime of host functions: memory the runtime knows (pinned by the caller, or not readable by the host) is
handed to hipMemcpy and never touched by the copying threads, everything else goes through the pinned slots."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# "Device" memory is ordinary memory of this process; an array at an address of `opaque` is one that only
# hipMemcpy can resolve (its pages cannot be read), kept in `behind`.
FAKE = r"""
#pragma once
#include <chrono>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorLaunchFailure = 719 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
struct hipPointerAttribute_t { hipMemoryType type; };
typedef void* hipStream_t;
enum { hipEventDisableTiming = 2, hipHostMallocDefault = 0 };
struct Pending { void* to; const void* from; size_t n; };
struct FakeEvent { std::vector<Pending> work; };
typedef FakeEvent* hipEvent_t;

struct Fake {
    std::mutex mu;
    std::vector<Pending> queue;  // copies since the last event
    const char *known = nullptr, *opaque = nullptr, *slow = nullptr;  // begins of special ranges
    size_t known_n = 0, opaque_n = 0, slow_n = 0;
    char* behind = nullptr;      // the opaque range's contents
    size_t direct = 0, staged = 0;  // bytes
    bool no_pinned = false;
};
inline Fake fake;
inline thread_local hipError_t fake_last = hipSuccess;
inline bool within(const void* p, const char* b, size_t n) {
    return b && (const char*)p >= b && (const char*)p < b + n;
}
inline void* resolve(const void* p) {
    return within(p, fake.opaque, fake.opaque_n) ? fake.behind + ((const char*)p - fake.opaque) : (void*)p;
}
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(resolve(d), resolve(s), n);
    std::lock_guard<std::mutex> lk(fake.mu);
    fake.direct += n;
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
    std::lock_guard<std::mutex> lk(fake.mu);
    fake.staged += n;
    if (k == hipMemcpyHostToDevice) std::memcpy(d, s, n);
    else fake.queue.push_back(Pending{d, s, n});
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { *e = new FakeEvent; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    std::lock_guard<std::mutex> lk(fake.mu);
    // (copies of other lanes queued before belong to earlier work of the same stream)
    for (const Pending& p : fake.queue) std::memcpy(p.to, p.from, p.n);
    e->work = fake.queue;
    fake.queue.clear();
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    for (const Pending& p : e->work)
        if (within(p.from, fake.slow, fake.slow_n)) std::this_thread::sleep_for(std::chrono::milliseconds(300));
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, int) {
    if (fake.no_pinned) return fake_last = hipErrorOutOfMemory;
    *p = std::malloc(n);
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
inline hipError_t hipGetLastError() { const hipError_t e = fake_last; fake_last = hipSuccess; return e; }
inline hipError_t hipPeekAtLastError() { return fake_last; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    a->type = within(p, fake.known, fake.known_n)     ? hipMemoryTypeHost
              : within(p, fake.opaque, fake.opaque_n) ? hipMemoryTypeDevice
                                                      : hipMemoryTypeUnregistered;
    return hipSuccess;
}
"""

MAIN = r"""
#include "zq3d_hostcopy.h"
#include <cstdio>
#include <sys/mman.h>
using namespace zq3d;
static const size_t N = 9u << 20;
static std::vector<char> array(int seed) {
    std::vector<char> v(N);
    for (size_t i = 0; i < N; i++) v[i] = (char)(i * 31 + i / 4093 + seed);
    return v;
}
static int failed(int line, const char* what) {
    return std::printf("line %d: %s (direct %zu staged %zu)\n", line, what, fake.direct, fake.staged), 1;
}
#define CHECK(c) do { if (!(c)) return failed(__LINE__, #c); } while (0)
int main() {
    HostCopy h;
    BODY
    h.release();
    std::printf("ok\n");
    return 0;
}
"""

# arrays pinned by the caller, and ordinary ones beside them, both ways
PINNED = r"""
    std::vector<char> a = array(1), b = array(2), da(N), db(N), a0 = a, b0 = b;
    fake.known = a.data(), fake.known_n = N;
    CHECK(h.to_device({{da.data(), a.data(), N}, {db.data(), b.data(), N}}) == hipSuccess);
    CHECK(da == a0 && db == b0 && fake.direct == N && fake.staged == N);
    CHECK(h.to_host({{db.data(), a.data(), N}, {da.data(), b.data(), N}}) == hipSuccess);
    CHECK(a == b0 && b == a0 && fake.direct == 2 * N && fake.staged == 2 * N);
"""
# an array whose pages the host cannot read
OPAQUE = r"""
    std::vector<char> a = array(3), b = array(4), da(N), db(N), hidden = a, b0 = b;
    void* p = mmap(nullptr, N, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    fake.opaque = (const char*)p, fake.opaque_n = N, fake.behind = hidden.data();
    CHECK(h.to_device({{da.data(), p, N}, {db.data(), b.data(), N}}) == hipSuccess);
    CHECK(da == a && db == b0);
    CHECK(h.to_host({{db.data(), p, N}, {da.data(), b.data(), N}}) == hipSuccess);
    CHECK(hidden == b0 && b == a);
"""
# two results for one array (a caller with one scalar field passes it twice): the later one stays, also where
# the earlier one's copies are slow to arrive
SHARED = r"""
    std::vector<char> host(2 * N), first = array(5), second = array(6);
    fake.slow = first.data(), fake.slow_n = 64;
    CHECK(h.to_host({{first.data(), host.data(), N}, {second.data(), host.data(), N}}) == hipSuccess);
    CHECK(std::memcmp(host.data(), second.data(), N) == 0);
    CHECK(h.to_host({{first.data(), host.data() + N / 2, N}, {second.data(), host.data(), N}}) == hipSuccess);
    CHECK(std::memcmp(host.data(), second.data(), N) == 0);
    CHECK(std::memcmp(host.data() + N, first.data() + N / 2, N / 2) == 0);
"""
# a kernel launch that failed before the copies is still reported when they find no pinned memory
FAILED_LAUNCH = r"""
    std::vector<char> host(N), dev = array(7);
    fake.no_pinned = true;
    fake_last = hipErrorLaunchFailure;
    hipError_t e = h.to_host({{dev.data(), host.data(), N}});
    if (e == hipSuccess) e = hipGetLastError();
    CHECK(e == hipErrorLaunchFailure && host == dev);
    fake_last = hipSuccess;
    CHECK(h.to_device({{dev.data(), host.data(), N}}) == hipSuccess && hipGetLastError() == hipSuccess);
"""


def run(tmp_path, body):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(FAKE)
    src = tmp_path / "copy.cpp"
    src.write_text(MAIN.replace("BODY", body))
    exe = str(tmp_path / "copy")
    inc = os.path.join(ROOT, "zq_smokesimulation_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", str(tmp_path), "-I", inc, str(src), "-o",
                    exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", (out.returncode, out.stdout)


@pytest.mark.parametrize("body", [PINNED, OPAQUE], ids=["pinned", "opaque"])
def test_memory_the_runtime_knows_goes_to_hipmemcpy(tmp_path, body):
    run(tmp_path, body)


def test_results_for_one_array_keep_their_order(tmp_path):
    run(tmp_path, SHARED)


def test_an_earlier_error_is_not_lost(tmp_path):
    run(tmp_path, FAILED_LAUNCH)
