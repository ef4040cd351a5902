"""The pool of closed sessions' device buffers, compiled for the host over a
memory of its own: hot sizes stay whatever was closed before them, idle
buffers stay within their bound and go back when an allocation fails, pooled
or direct."""
import os
import subprocess

from conftest import ROOT

DRIVER = r"""
#include <cassert>
#include <cstdint>
#include <set>
#include <thread>
#include <vector>
#include "xpu_devpool.h"

struct Mem
{
    typedef int Error;
    static constexpr int OUT_OF_MEMORY = 2;
    static std::mutex m;
    static std::map<void *, size_t> held;
    static size_t used, limit;
    static uintptr_t next;
    static int calls;
    static int device() { return dev; }
    static int dev;
    static int alloc(void **p, size_t n)
    {
        std::lock_guard<std::mutex> g(m);
        calls++;
        if (used + n > limit)
            return OUT_OF_MEMORY;
        *p = (void *)(next += 1 << 20);
        held[*p] = n;
        used += n;
        return 0;
    }
    static void release(void *p)
    {
        std::lock_guard<std::mutex> g(m);
        assert(held.count(p));
        used -= held[p];
        held.erase(p);
    }
};
std::mutex Mem::m;
std::map<void *, size_t> Mem::held;
size_t Mem::used = 0, Mem::limit = 64ULL << 30;
uintptr_t Mem::next = 0;
int Mem::calls = 0, Mem::dev = 0;

typedef DevPool<Mem> Pool;
static const size_t GB = 1ULL << 30, MB = 1ULL << 20;

static void *
get(Pool &P, size_t n)
{
    void *p = nullptr;
    assert(P.alloc(&p, n) == 0);
    assert(Mem::held.at(p) >= n);
    return p;
}

/* eight idle buffers of 1 GiB fill the pool; a size used afterwards is kept */
static void
hot_size_stays()
{
    Pool P;
    std::vector<void *> old;
    for (int i = 0; i < 8; i++)
        old.push_back(get(P, GB));
    for (void *p : old)
        P.free(p);
    const int before = Mem::calls;
    for (int i = 0; i < 10; i++)
    {
        void *a = get(P, 300 * MB), *b = get(P, 90 * MB);
        P.free(a);
        P.free(b);
    }
    assert(Mem::calls == before + 2);
    assert(Mem::used <= XPU_POOL_BYTES);
    P.trim();
    assert(Mem::used == 0 && P.idle_bytes == 0);
}

/* the oldest goes first, and no more than is needed */
static void
oldest_goes_first()
{
    Pool P;
    std::vector<void *> v;
    for (int i = 0; i < 9; i++)
        v.push_back(get(P, (900 + i) * MB));
    for (void *p : v)
        P.free(p);
    assert(Mem::held.size() == 8 && !Mem::held.count(v[0]) && Mem::held.count(v[1]));
    void *big = get(P, 9 * GB);             /* never kept */
    P.free(big);
    assert(!Mem::held.count(big) && Mem::held.size() == 8);
    for (int i = 0; i < 1100; i++)
        v.push_back(get(P, 256));
    for (size_t i = 9; i < v.size(); i++)
        P.free(v[i]);
    assert(Mem::held.size() == XPU_POOL_COUNT);
    P.trim();
    assert(Mem::used == 0);
}

/* a buffer up to a quarter larger is taken, a larger one and another device's
 * are not */
static void
near_sizes()
{
    Pool P;
    void *a = get(P, 120 * MB);
    P.free(a);
    assert(get(P, 100 * MB) == a);
    P.free(a);
    void *b = get(P, 80 * MB);
    assert(b != a);
    Mem::dev = 1;
    void *c = get(P, 120 * MB);
    assert(c != a);
    Mem::dev = 0;
    assert(get(P, 120 * MB) == a);
    P.free(a);
    P.free(b);
    P.free(c);
    P.trim();
    assert(Mem::used == 0);
}

/* what is idle goes back when the device has no room: for the pool's own
 * buffers and for those outside it; what is in use stays */
static void
room_on_failure()
{
    Pool P;
    Mem::limit = 6 * GB;
    void *keep = get(P, GB), *a = get(P, 2 * GB), *b = get(P, 2 * GB);
    P.free(a);
    P.free(b);
    void *p = nullptr;
    assert(P.alloc_direct(&p, 4 * GB) == 0);
    assert(Mem::held.count(keep) && Mem::held.size() == 2);
    Mem::release(p);
    P.free(get(P, 4 * GB));
    void *q = get(P, 5 * GB);
    assert(P.alloc(&p, 5 * GB) == Mem::OUT_OF_MEMORY);
    P.free(q);
    P.free(keep);
    P.trim();
    assert(Mem::used == 0);
    Mem::limit = 64 * GB;
}

static void
threads()
{
    Pool P;
    std::vector<std::thread> t;
    for (int k = 0; k < 8; k++)
        t.emplace_back([&P, k] {
            for (int i = 0; i < 2000; i++)
            {
                void *a = nullptr, *b = nullptr;
                assert(P.alloc(&a, (1 + (i * 7 + k) % 40) * 50 * MB) == 0);
                assert(P.alloc(&b, 1000 + i) == 0 && a != b);
                P.free(a);
                if (i % 97 == 0)
                    P.trim();
                P.free(b);
            }
        });
    for (auto &x : t)
        x.join();
    P.trim();
    assert(Mem::used == 0 && P.live.empty());
}

int
main()
{
    assert(Pool::round_up(0) == 256 && Pool::round_up(1) == 256 && Pool::round_up(257) == 512);
    for (size_t n = 2048; n < 100000; n += 37)
        assert(Pool::round_up(n) >= n && Pool::round_up(n) <= n + n / 8);
    hot_size_stays();
    oldest_goes_first();
    near_sizes();
    room_on_failure();
    threads();
    return 0;
}
"""


def test_pool(tmp_path):
    src = tmp_path / "pool.cpp"
    src.write_text(DRIVER)
    exe = tmp_path / "pool"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread",
                    "-I" + os.path.join(ROOT, "pg-strom_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    subprocess.run([str(exe)], check=True, timeout=120)
