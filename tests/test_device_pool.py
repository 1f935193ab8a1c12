"""The pool of destroyed solvers' memory (cedar_amd/csrc/device_pool.cpp), built with the host compiler
against a HIP runtime of a few lines that counts what is allocated: limit, eviction, trim, the retry
after a failed allocation, blocks that are not idle, several threads."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cedar_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <cstddef>
#include <cstdlib>
#include <map>
#include <mutex>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone, hipStreamCaptureStatusActive };
enum { hipStreamNonBlocking = 1 };
struct fake_stream { int device; };
using hipStream_t = fake_stream *;
namespace fake {
inline std::mutex mu;
inline std::map<void *, std::size_t> blocks;
inline std::size_t used = 0, room = ~std::size_t(0);
inline int streams = 0;
inline bool busy = false, capturing = false;  // busy: waiting fails
inline thread_local int device = 0;
}
inline hipError_t hipGetDevice(int *d) { *d = fake::device; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipMalloc(void **p, std::size_t n) {
    std::lock_guard<std::mutex> g(fake::mu);
    if (fake::used + n > fake::room) { *p = nullptr; return hipErrorOutOfMemory; }
    *p = std::malloc(1);
    fake::blocks[*p] = n;
    fake::used += n;
    return hipSuccess;
}
inline hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> g(fake::mu);
    const auto it = fake::blocks.find(p);
    if (it == fake::blocks.end()) std::abort();  // freed twice
    fake::used -= it->second;
    fake::blocks.erase(it);
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return fake::busy ? hipErrorUnknown : hipSuccess; }
inline hipError_t hipStreamCreateWithFlags(hipStream_t *s, int) {
    *s = new fake_stream{fake::device};
    ++fake::streams;
    return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) { delete s; --fake::streams; return hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, int *d) { *d = s->device; return hipSuccess; }
inline hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *st) {
    *st = fake::capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
"""

PROGRAM = r"""
#include "device_pool.hpp"
#include <cstdio>
#include <thread>
#include <vector>
using namespace cedar::hip;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
static void *get(std::size_t n) { hipError_t e; return pool_malloc(n, &e); }
static void give(void *p) { pool_idle_scope s(nullptr); pool_free(p); }
int main() {
    const std::size_t K = 1024, first = pool_set_limit(8 * K);
    std::printf("%zu\n", first);
    // kept, handed out again, and only to the same size and device
    void *a = get(2 * K);
    give(a);
    CHECK(fake::used == 2 * K);
    fake::device = 1;
    void *d = get(2 * K);
    CHECK(d != a);
    pool_free(d);
    fake::device = 0;
    void *c = get(K);
    CHECK(c != a && get(2 * K) == a);
    // not idle: outside a scope, of another device, where the stream cannot be waited for (inside a
    // scope of another stream too), and where the caller has been given pointers
    pool_free(c);
    CHECK(fake::used == 2 * K);
    { pool_idle_scope s(nullptr); fake::device = 1; void *o = get(K); pool_free(o); fake::device = 0; }
    CHECK(fake::used == 2 * K);
    fake::busy = true;
    give(a);
    fake::busy = false;
    CHECK(fake::used == 0);
    a = get(K);
    {
        pool_idle_scope s(nullptr);
        fake::busy = true;
        give(a);
        fake::busy = false;
        CHECK(fake::used == 0);
        pool_free(get(K));  // the outer scope holds again
        CHECK(fake::used == K && pool_trim() == K);
    }
    for (bool lent : {true, false}) {
        void *p = get(K);
        pool_guard guard;
        if (lent) guard.lend();
        guard.enter(nullptr);
        pool_free(p);
        CHECK(fake::used == (lent ? 0 : K));
    }
    CHECK(pool_trim() == K);
    // captured: nothing is kept, nor by a guard that is destroyed inside
    for (bool captured : {true, false}) {
        void *outer = get(K), *inner = get(2 * K);
        pool_guard guard;
        fake::capturing = captured;
        guard.lend_if_captured(nullptr);
        fake::capturing = false;
        guard.enter(nullptr);
        {
            pool_guard g2;
            g2.enter(nullptr);
            pool_free(inner);
        }
        pool_free(outer);
        CHECK(fake::used == (captured ? 0 : 3 * K));
    }
    CHECK(pool_trim() == 3 * K);
    give(get(K));
    CHECK(pool_trim() == K);
    // the ones kept longest go beyond the limit; one larger than it is never kept
    std::vector<void *> v;
    for (int i = 0; i < 5; ++i) v.push_back(get(2 * K));
    for (void *p : v) give(p);
    CHECK(fake::used == 8 * K && !fake::blocks.count(v[0]) && fake::blocks.count(v[4]));
    give(get(9 * K));
    CHECK(fake::used == 8 * K);
    // lowering the limit gives back what lies beyond; live blocks stay
    void *live = get(2 * K);
    CHECK(pool_set_limit(4 * K) == 8 * K && fake::used == 6 * K);
    CHECK(pool_set_limit(0) == 4 * K && fake::used == 2 * K);
    give(live);
    CHECK(fake::used == 0);
    // trim gives everything back, streams too
    pool_set_limit(8 * K);
    hipError_t e;
    hipStream_t s = pool_capture_stream(&e);
    pool_return_capture_stream(s);
    CHECK(fake::streams == 1);
    live = get(K);
    give(get(3 * K));
    give(get(K));
    CHECK(pool_trim() == 4 * K && fake::used == K && fake::streams == 0 && pool_trim() == 0);
    give(live);
    pool_trim();
    // an allocation that fails is tried again without the kept blocks, and fails if that is no help
    fake::room = 8 * K;
    give(get(5 * K));
    void *big = pool_malloc(7 * K, &e);
    CHECK(big && e == hipSuccess && fake::used == 7 * K);
    CHECK(!pool_malloc(2 * K, &e) && e == hipErrorOutOfMemory);
    give(big);
    fake::room = ~std::size_t(0);
    pool_trim();
    // threads: every block is one thread's at a time, and all come back
    bool bad = false;
    auto work = [&](int t) {
        for (int r = 0; r < 2000; ++r) {
            std::vector<void *> mine;
            for (int i = 0; i < 4; ++i) {
                void *p = get((i % 2 + 1) * K);
                *static_cast<char *>(p) = (char)t;
                mine.push_back(p);
            }
            for (void *p : mine) bad |= *static_cast<char *>(p) != (char)t;
            for (void *p : mine) give(p);
            if (r % 100 == 0) pool_trim();
        }
    };
    std::vector<std::thread> ts;
    for (int t = 0; t < 4; ++t) ts.emplace_back(work, t);
    for (auto &t : ts) t.join();
    pool_trim();
    CHECK(!bad && fake::used == 0 && fake::blocks.empty());
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("pool")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (d / "main.cpp").write_text(PROGRAM)
    r = subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-pthread", f"-I{d}", f"-I{CSRC}",
                        str(d / "main.cpp"), os.path.join(CSRC, "device_pool.cpp"), "-o",
                        str(d / "pool")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return str(d / "pool")


# the limit that the environment sets, and what is no number of MiB sets none
@pytest.mark.parametrize("value,limit", [(None, 4 << 30), ("0", 0), ("17", 17 << 20), ("", 4 << 30),
                                         ("1x", 4 << 30), ("-1", 4 << 30)])
def test_pool(program, value, limit):
    env = {k: v for k, v in os.environ.items() if k != "CEDAR_AMD_POOL_MB"}
    if value is not None:
        env["CEDAR_AMD_POOL_MB"] = value
    r = subprocess.run([program], capture_output=True, text=True, env=env, timeout=60)
    assert r.returncode == 0, r.stdout
    assert r.stdout.split() == [str(limit)]
