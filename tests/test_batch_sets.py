"""The idle batch buffers of a model (kvd_batch.h), compiled for the host against
a counted device of its own: which set a call takes, the bound on idle ones, and
that an allocation on a full device frees idle sets instead of failing."""
import os
import shutil
import subprocess

import pytest

HDR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "shannon-prime-system_amd", "csrc", "hip", "kvd_batch.h")
PRE = """#include <algorithm>
#include <cassert>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstdio>
#include <map>
#include <mutex>
#include <thread>
#include <vector>
#undef NDEBUG
struct int2 { int x, y; };
enum hipError_t { hipSuccess, hipErrorOutOfMemory, hipErrorInvalidValue };
typedef struct Event *hipEvent_t;
static std::mutex dmu;
static size_t room = 100, fails = 0;
static hipError_t last = hipSuccess;
static std::map<void *, size_t> held;
static hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::mutex> lk(dmu);
    if (n > room) { fails++; return last = hipErrorOutOfMemory; }
    room -= n; *p = malloc(1); held[*p] = n;
    return hipSuccess;
}
static hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> lk(dmu);
    assert(held.count(p));
    room += held[p]; held.erase(p); free(p);
    return hipSuccess;
}
static hipError_t hipHostFree(void *) { return hipSuccess; }
static hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
static hipError_t hipGetLastError() { hipError_t e = last; last = hipSuccess; return e; }
"""
MAIN = """
using namespace kvd;
static Batch lease(BatchSets &s, bool flt, int pmax, size_t bytes) {
    Batch b = s.take(flt, pmax);
    if (!b.buf) { assert(dev_malloc(&b.buf, bytes) == hipSuccess); b.bytes = bytes; }
    return b;
}
int main() {
    {
        BatchSets s, other;
        // the smallest set that serves the call; float sets serve both modes
        Batch big = lease(s, true, 4096, 40), mid = lease(s, false, 4096, 20), small = lease(s, false, 64, 5);
        assert(room == 35 && big.flt && big.pmax == 4096 && !small.flt && small.pmax == 64);
        void *pb = big.buf, *pm = mid.buf, *ps = small.buf;
        s.give(big); s.give(small); s.give(mid);
        Batch a = s.take(false, 64), b = s.take(false, 64), c = s.take(false, 64), d = s.take(false, 64);
        assert(a.buf == ps && b.buf == pm && c.buf == pb && !d.buf && d.pmax == 64);
        s.give(c); s.give(a); s.give(b);
        a = s.take(false, 65); b = s.take(true, 64);
        assert(a.buf == pm && b.buf == pb && !s.take(true, 1).buf && !s.take(false, 65).buf);
        s.give(a); s.give(b);
        // a full device: idle sets go, of every model, and the allocation succeeds
        // with no error left behind; without idle sets it fails as it did
        Batch o = lease(other, false, 64, 30);
        other.give(o);
        void *p = nullptr, *q = nullptr;
        assert(room == 5 && dev_malloc(&p, 100) == hipSuccess && room == 0 && last == hipSuccess && fails == 1);
        assert(dev_malloc(&q, 1) == hipErrorOutOfMemory && fails == 2 && hipGetLastError() == hipErrorOutOfMemory);
        assert(!s.take(false, 1).buf);
        hipFree(p);
        // a set in use is nobody's to free
        a = lease(s, false, 64, 60);
        assert(dev_malloc(&q, 50) == hipErrorOutOfMemory && held.size() == 1);
        s.give(a);
        // at most MAX_IDLE_BATCHES idle: the oldest goes
        assert(BatchSets::reclaim() && !BatchSets::reclaim() && room == 100);
        std::vector<Batch> v;
        for (int i = 0; i < 6; i++) v.push_back(lease(s, false, 100 + i, 1));
        for (Batch &x : v) s.give(x);
        assert(room == 100 - MAX_IDLE_BATCHES && s.take(false, 0).pmax == 102);
        v[2].release();
        last = hipSuccess;
    }
    assert(room == 100 && held.empty());       // a model's end frees the rest
    {
        BatchSets s, t;
        std::vector<std::thread> th;
        for (int k = 0; k < 8; k++)
            th.emplace_back([&, k] {
                for (int i = 0; i < 2000; i++) {
                    BatchSets &m = k & 1 ? s : t;
                    Batch b = m.take(i % 3 == 0, i % 7);
                    if (!b.buf) { if (dev_malloc(&b.buf, 11) != hipSuccess) continue; b.bytes = 11; }
                    if (i % 5) m.give(b); else b.release();
                }
            });
        for (auto &x : th) x.join();
    }
    assert(room == 100 && held.empty());
    return 0;
}
"""


def test_idle_sets(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ is not installed")
    body = "".join(line for line in open(HDR) if not line.startswith(("#include", "#pragma once")))
    (tmp_path / "b.cpp").write_text(PRE + body + MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-w", "-pthread",
                    str(tmp_path / "b.cpp"), "-o", str(tmp_path / "b")], check=True)
    env = {k: v for k, v in os.environ.items() if k != "LD_PRELOAD"}
    r = subprocess.run([str(tmp_path / "b")], env=env, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
