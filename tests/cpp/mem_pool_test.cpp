// The build memory pool (vkhrt_amd/csrc/mem_pool.hpp) over a counted stand-in for the HIP allocator:
// reuse, eviction, memory running out in a pool, in another context's pool and in the library's
// other allocations, closing, and blocks passed between threads. Host C++, no GPU.
#include <stdio.h>
#include <stdlib.h>

#include <map>
#include <thread>
#include <vector>

#include "../../vkhrt_amd/csrc/mem_pool.hpp"

namespace {
std::mutex g_m;
std::map<void*, std::pair<size_t, int>> g_live;  // size and device
size_t g_used[2], g_limit[2] = {size_t(1) << 40, size_t(1) << 40};
thread_local int g_device;
uintptr_t g_next = 4096;

#define CHECK(x)                                                     \
    do {                                                             \
        if (!(x)) {                                                  \
            fprintf(stderr, "line %d: %s\n", __LINE__, #x);          \
            exit(1);                                                 \
        }                                                            \
    } while (0)

constexpr size_t MiB = size_t(1) << 20;
using vk::MemPool;

MemPool::Block get(MemPool& p, size_t bytes) {
    MemPool::Block b;
    CHECK(p.acquire(bytes, &b) == hipSuccess && b.p && b.bytes >= bytes);
    return b;
}
size_t live() { return g_live.size(); }
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> g(g_m);
    if (g_used[g_device] + bytes > g_limit[g_device]) return hipErrorOutOfMemory;
    g_used[g_device] += bytes;
    *p = reinterpret_cast<void*>(g_next);
    g_next += bytes + 4096;
    g_live[*p] = {bytes, g_device};
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> g(g_m);
    if (!p) return hipSuccess;
    auto it = g_live.find(p);
    CHECK(it != g_live.end());  // freed once
    g_used[it->second.second] -= it->second.first;
    g_live.erase(it);
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = g_device;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
}

int main() {
    {  // a block comes back for the same size and up to a quarter less, not for more or much less
        MemPool p(0);
        MemPool::Block a = get(p, 8 * MiB);
        void* first = a.p;
        p.release(a, true);
        CHECK(live() == 1);
        a = get(p, 7 * MiB);
        CHECK(a.p == first && a.bytes == 8 * MiB);
        void* fence = nullptr;
        CHECK(MemPool::make_fence(&fence) == hipSuccess && live() == 2);
        p.release(a, MemPool::wait(fence));
        CHECK(live() == 1);
        a = get(p, 8 * MiB);
        CHECK(a.p == first && !MemPool::wait(nullptr));
        p.release(a, false);  // perhaps in use: not kept
        CHECK(live() == 0);
        a = get(p, 8 * MiB);
        first = a.p;
        p.release(a, true);
        MemPool::Block b = get(p, 9 * MiB), c = get(p, 4 * MiB);
        CHECK(b.p != first && c.p != first && live() == 3);
        p.release(b, true);
        p.release(c, true);
        MemPool::Block s = get(p, MiB / 2);  // small blocks are not kept
        p.release(s, true);
        CHECK(live() == 3);
    }
    CHECK(live() == 0);
    {  // at most 8 blocks: the one kept longest goes
        MemPool p(0);
        std::vector<MemPool::Block> v;
        for (int i = 0; i < 10; ++i) v.push_back(get(p, (2 << i) * MiB / 4 + 2 * MiB));
        for (auto& b : v) p.release(b, true);
        CHECK(live() == 8 && !g_live.count(v[0].p) && !g_live.count(v[1].p) && g_live.count(v[2].p));
    }
    {  // at most 1 GiB: as many of the oldest go as make room; a larger block is not kept
        MemPool p(0);
        MemPool::Block a = get(p, 300 * MiB), b = get(p, 400 * MiB), c = get(p, 500 * MiB), d = get(p, 1025 * MiB);
        p.release(a, true);
        p.release(b, true);
        p.release(c, true);
        CHECK(!g_live.count(a.p) && g_live.count(b.p) && g_live.count(c.p));
        p.release(d, true);
        CHECK(!g_live.count(d.p) && live() == 2);
    }
    CHECK(live() == 0);
    {  // memory runs out while blocks are kept: they are freed and the allocation succeeds, in the pool
       // itself, in another context's pool and in an allocation that is not a pool's
        MemPool p(0), q(0), other(1);
        g_limit[0] = 1000 * MiB;
        auto keep = [&] {
            g_device = 0;
            p.release(get(p, 600 * MiB), true);
            CHECK(g_used[0] == 600 * MiB);
        };
        g_device = 1;
        other.release(get(other, 100 * MiB), true);
        keep();
        MemPool::Block a = get(p, 900 * MiB);
        p.release(a, true);
        CHECK(g_used[0] == 900 * MiB);
        p.trim();
        keep();
        a = get(q, 900 * MiB);
        q.release(a, true);
        q.trim();
        keep();
        float* buf = nullptr;
        CHECK(vk::device_malloc(&buf, 900 * MiB) == hipSuccess && g_used[0] == 900 * MiB);
        (void)hipFree(buf);
        CHECK(g_used[1] == 100 * MiB);  // another device's memory stays
        CHECK(vk::device_malloc(&buf, 1001 * MiB) == hipErrorOutOfMemory);
        CHECK(p.acquire(1001 * MiB, &a) == hipErrorOutOfMemory && !a.p);
        g_limit[0] = size_t(1) << 40;
    }
    CHECK(live() == 0);
    {  // a closed pool keeps nothing, and takes back what outlives its context
        MemPool p(0);
        MemPool::Block a = get(p, 8 * MiB), b = get(p, 8 * MiB);
        p.release(a, true);
        p.close();
        CHECK(live() == 1);
        p.release(b, false);
        CHECK(live() == 0);
    }
    {  // blocks passed between threads have one owner at a time, while another thread runs out of memory
        MemPool p(0), q(0);
        std::mutex m;
        std::map<void*, int> owner;
        std::vector<std::thread> threads;
        for (int t = 0; t < 6; ++t)
            threads.emplace_back([&, t] {
                unsigned r = unsigned(t) * 7919u + 1u;
                for (int i = 0; i < 3000; ++i) {
                    MemPool& pool = (r >> 20) & 1u ? p : q;
                    r = r * 1664525u + 1013904223u;
                    MemPool::Block b = get(pool, (1 + (r >> 16) % 64) * MiB);
                    {
                        std::lock_guard<std::mutex> g(m);
                        CHECK(owner.emplace(b.p, t).second);
                    }
                    if (t == 0 && i % 50 == 0)
                        CHECK(MemPool::retry_trimmed([] { return hipErrorOutOfMemory; }) == hipErrorOutOfMemory);
                    {
                        std::lock_guard<std::mutex> g(m);
                        owner.erase(b.p);
                    }
                    pool.release(b, (r >> 8) & 1u);
                }
            });
        for (auto& t : threads) t.join();
        CHECK(live() <= 16);
    }
    CHECK(live() == 0);
    printf("mem_pool ok\n");
    return 0;
}
