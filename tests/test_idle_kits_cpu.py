"""CPU: the streams and pinned pages that destroyed handles leave to the next ones, and the no-allocation call's
page (miniisosurface_amd/csrc/idle_kits.h), compiled against a small HIP runtime of this test's own that counts
what is alive, gives recycled handles and addresses, can refuse a call, leave a stream unfinished and reset its
device: nothing is lost, nothing is handed on or freed that a reset took away, at most four wait per device."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = os.environ.get("CXX", "g++")

RUNTIME = r"""
#pragma once
#include <cstdint>
#include <map>
#include <mutex>
#include <set>
typedef enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorNotReady = 600 } hipError_t;
typedef struct Stream_* hipStream_t;
typedef void* hipDeviceptr_t;
enum { hipStreamDefault = 0, hipHostMallocDefault = 0 };
typedef enum { hipStreamCaptureModeGlobal, hipStreamCaptureModeThreadLocal, hipStreamCaptureModeRelaxed } hipStreamCaptureMode;
typedef enum { HIP_POINTER_ATTRIBUTE_BUFFER_ID } hipPointer_attribute;
struct Fake {
    std::mutex m;
    int dev = 0;
    std::set<uintptr_t> free_addresses;            // the lowest one is given out next: recycled at once
    uintptr_t next = 0x1000;
    std::map<uintptr_t, int> streams;              // handle -> device
    std::map<uintptr_t, std::pair<int, unsigned long long>> memory;   // address -> device (-1 host), id
    unsigned long long ids = 0;
    bool busy = false, no_ids = false;
    int wrong = 0;                                 // frees of what is not there
    int refuse_stream = 0, refuse_host = 0, refuse_device = 0, host_calls = 0;
    uintptr_t address()
    {
        uintptr_t a = next;
        if (free_addresses.empty()) next += 0x1000;
        else { a = *free_addresses.begin(); free_addresses.erase(free_addresses.begin()); }
        return a;
    }
};
inline Fake& fake() { static Fake* f = new Fake; return *f; }
#define HELD Fake& f = fake(); std::lock_guard<std::mutex> held(f.m)
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = fake().dev; return hipSuccess; }
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    HELD;
    if (f.refuse_stream) return hipErrorOutOfMemory;
    const uintptr_t a = f.address();
    f.streams[a] = f.dev;
    *s = (hipStream_t)a;
    return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s)
{
    HELD;
    if (!f.streams.erase((uintptr_t)s)) { ++f.wrong; return hipErrorInvalidValue; }
    f.free_addresses.insert((uintptr_t)s);
    return hipSuccess;
}
inline hipError_t hipStreamQuery(hipStream_t s)
{
    HELD;
    return !f.streams.count((uintptr_t)s) ? hipErrorInvalidValue : f.busy ? hipErrorNotReady : hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { fake().busy = false; return hipSuccess; }
inline hipError_t alloc(void** p, int dev)
{
    Fake& f = fake();
    const uintptr_t a = f.address();
    f.memory[a] = {dev, ++f.ids};
    *p = (void*)a;
    return hipSuccess;
}
inline hipError_t hipMalloc(void** p, size_t) { HELD; return f.refuse_device ? hipErrorOutOfMemory : alloc(p, f.dev); }
inline hipError_t hipHostMalloc(void** p, size_t, unsigned) { HELD; ++f.host_calls; return f.refuse_host ? hipErrorOutOfMemory : alloc(p, -1); }
inline hipError_t hipFree(void* p)
{
    HELD;
    if (!f.memory.erase((uintptr_t)p)) { ++f.wrong; return hipErrorInvalidValue; }
    f.free_addresses.insert((uintptr_t)p);
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) { return hipFree(p); }
inline hipError_t hipPointerGetAttribute(void* out, hipPointer_attribute, hipDeviceptr_t p)
{
    HELD;
    const auto it = f.memory.find((uintptr_t)p);
    if (f.no_ids || it == f.memory.end()) return hipErrorInvalidValue;
    *(unsigned long long*)out = it->second.second;
    return hipSuccess;
}
inline void reset_device(int dev)
{
    HELD;
    for (auto it = f.streams.begin(); it != f.streams.end();)
        if (it->second == dev) { f.free_addresses.insert(it->first); it = f.streams.erase(it); } else ++it;
    for (auto it = f.memory.begin(); it != f.memory.end();)
        if (it->second.first == dev || it->second.first == -1) { f.free_addresses.insert(it->first); it = f.memory.erase(it); } else ++it;
}
#undef HELD
"""

PROGRAM = r"""
#include "idle_kits.h"
#include <cstdio>
#include <cstring>
#include <thread>
#include <vector>
using namespace miso;
#define EXPECT(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
static size_t alive() { return fake().streams.size() + fake().memory.size(); }
static std::vector<Kit> take(int n)
{
    std::vector<Kit> k(n);
    for (Kit& q : k)
        if (idle_kits().take(&q) != hipSuccess) q = Kit();
    return k;
}
int main(int, char** argv)
{
    const char* what = argv[1];
    Fake& f = fake();
    if (!strcmp(what, "bounded")) {
        for (int round = 0; round < 3; ++round) {
            auto k = take(9);
            for (auto& a : k) for (auto& b : k) EXPECT(&a == &b || (a.stream != b.stream && a.totals != b.totals));
            for (auto& q : k) { idle_kits().leave(q, true); EXPECT(!q.stream && !q.totals); }
            EXPECT(f.streams.size() == 4);
        }
        f.dev = 3;                                  // another device has its own
        auto k = take(2);
        EXPECT(f.streams.size() == 6);
        f.dev = 0;
        for (auto& q : k) idle_kits().leave(q, true);
        EXPECT(f.streams.size() == 6);
        auto l = take(4);
        for (auto& q : l) EXPECT(q.dev == 0 && f.streams[(uintptr_t)q.stream] == 0);
        for (auto& q : l) idle_kits().leave(q, false);     // not clean: destroyed
        EXPECT(f.streams.size() == 2 && f.wrong == 0);
    } else if (!strcmp(what, "busy")) {             // a stream that still works, on the null stream's behalf
        auto k = take(1);
        const hipStream_t s = k[0].stream;
        idle_kits().leave(k[0], true);
        const size_t was = alive();
        for (int t = 0; t < 10; ++t) {
            f.busy = true;
            auto l = take(1);
            EXPECT(l[0].stream == s && alive() == was);
            idle_kits().leave(l[0], true);
        }
        EXPECT(alive() == was && f.wrong == 0);
    } else if (!strcmp(what, "reset")) {            // the new streams and pages have the old ones' handles
        auto k = take(3);
        for (auto& q : k) idle_kits().leave(q, true);
        reset_device(0);
        EXPECT(alive() == 0);
        std::vector<hipStream_t> theirs(9);
        std::vector<void*> mem(9);
        for (auto& s : theirs) hipStreamCreateWithFlags(&s, 0);
        for (auto& m : mem) hipMalloc(&m, 1);
        auto l = take(4);
        for (auto& q : l) {
            for (auto s : theirs) EXPECT(q.stream != s);
            for (auto m : mem) EXPECT((void*)q.totals != m);
            EXPECT(f.streams.count((uintptr_t)q.stream) && f.memory.count((uintptr_t)q.totals));
        }
        for (auto& q : l) idle_kits().leave(q, true);
        for (auto s : theirs) EXPECT(f.streams.count((uintptr_t)s));
        EXPECT(f.wrong == 0);
    } else if (!strcmp(what, "reset alive")) {      // a handle's end after a reset frees nothing of the new owner's
        auto k = take(1);
        reset_device(0);
        std::vector<hipStream_t> theirs(9);
        for (auto& s : theirs) hipStreamCreateWithFlags(&s, 0);
        const size_t was = alive();
        idle_kits().leave(k[0], true);
        EXPECT(alive() == was && f.wrong == 0);
        auto l = take(1);
        for (auto s : theirs) EXPECT(l[0].stream != s);
    } else if (!strcmp(what, "refused")) {
        int* const refuse[3] = {&f.refuse_stream, &f.refuse_host, &f.refuse_device};
        for (int* r : refuse) {
            *r = 1;
            Kit k;
            EXPECT(idle_kits().take(&k) == hipErrorOutOfMemory && !k.stream && alive() == 0);
            *r = 0;
        }
        EXPECT(f.wrong == 0);
    } else if (!strcmp(what, "no ids")) {           // nothing can be told from its successor: nothing is kept
        f.no_ids = true;
        auto k = take(2);
        for (auto& q : k) { EXPECT(q.stream && q.totals); idle_kits().leave(q, true); }
        EXPECT(alive() == 0 && f.wrong == 0);
        KeptPage page;
        EXPECT(!page.get() && alive() == 0);
    } else if (!strcmp(what, "threads")) {
        std::vector<std::thread> t;
        for (int n = 0; n < 8; ++n)
            t.emplace_back([] {
                for (int r = 0; r < 2000; ++r) {
                    auto k = take(1 + r % 3);
                    for (auto& q : k) idle_kits().leave(q, r % 7 != 0);
                }
            });
        for (auto& q : t) q.join();
        EXPECT(f.streams.size() <= 4 && alive() == 3 * f.streams.size() && f.wrong == 0);
    } else if (!strcmp(what, "page")) {
        KeptPage page;
        f.refuse_host = 1;
        EXPECT(!page.get());
        f.refuse_host = 0;
        uint64_t* p = page.get();                   // a later call tries again
        EXPECT(p && f.host_calls == 2);
        for (int t = 0; t < 5; ++t) EXPECT(page.get() == p);
        EXPECT(f.host_calls == 2);
        reset_device(0);
        void* theirs = nullptr;
        hipHostMalloc(&theirs, 1, 0);
        EXPECT(theirs == (void*)p);                 // the address is someone else's now
        uint64_t* q = page.get();
        EXPECT(q && q != p && page.get() == q && f.wrong == 0 && f.memory.size() == 2);
    } else {
        return 2;
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which(CXX):
        pytest.skip("no C++ compiler")
    tmp = tmp_path_factory.mktemp("kits")
    (tmp / "hip").mkdir()
    (tmp / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp / "kits.cpp").write_text(PROGRAM)
    exe = str(tmp / "kits")
    subprocess.run([CXX, "-O1", "-std=c++17", "-pthread", f"-I{tmp}",
                    "-I", os.path.join(ROOT, "miniisosurface_amd", "csrc"), "-o", exe, str(tmp / "kits.cpp")], check=True,
                   capture_output=True, text=True, timeout=120)
    return exe


@pytest.mark.parametrize("what", ["bounded", "busy", "reset", "reset alive", "refused", "no ids", "threads", "page"])
def test_idle_kits(program, what):
    out = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
