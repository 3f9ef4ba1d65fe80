// The workspace pool against counted memory: repeated calls of mixed sizes allocate once, what
// stays idle is bounded, the longest idle block makes room, devices and threads keep apart.
#include "runtime/workspace.h"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <thread>
#include <vector>

static std::atomic<int> g_allocs{0}, g_fail{0};
static std::atomic<long> g_held{0};
static thread_local int g_dev = 0;
static std::mutex g_mu;
static std::set<void*> g_live;

struct Counted {
    static bool device(int* dev) { *dev = g_dev; return g_dev >= 0; }
    static void* alloc(size_t bytes) {
        if (g_fail > 0) { g_fail--; return nullptr; }
        g_allocs++;
        g_held += (long)bytes;
        size_t* p = (size_t*)std::malloc(sizeof(size_t));
        *p = bytes;
        std::lock_guard<std::mutex> g(g_mu);
        g_live.insert(p);
        return p;
    }
    static bool free(void* p) {
        std::lock_guard<std::mutex> g(g_mu);
        if (!g_live.erase(p)) std::abort();
        g_held -= (long)*(size_t*)p;
        std::free(p);
        return true;
    }
};
using Pool = gpumpi::WorkspacePool<Counted>;

#define CHECK(x) if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; }

int main() {
    constexpr size_t MiB = 1u << 20;
    for (size_t need : {size_t(0), size_t(1), size_t(65536), size_t(65537), size_t(1000003), 35700000ul, 64 * MiB - 1, 64 * MiB, 64 * MiB + 1}) {
        const size_t r = Pool::rounded(need);
        CHECK(r >= need && (need > 64 * MiB ? r == need : r <= 64 * MiB && (r <= 65536 || r - need <= need / 8 + 1)));
    }
    Pool p;
    // a large bucket sort's two calls, a small one's between them
    for (int i = 0; i < 5; i++)
        for (size_t need : {35700000ul, 16800000ul, 70000ul}) {
            const Pool::Block b = p.take(need);
            CHECK(b.ptr && b.bytes >= need);
            p.give(b);
        }
    CHECK(g_allocs == 1);
    // two at a time: a block each, kept from then on
    for (int i = 0; i < 5; i++) {
        const Pool::Block a = p.take(35700000), b = p.take(16800000);
        CHECK(a.ptr != b.ptr);
        p.give(a);
        p.give(b);
    }
    CHECK(g_allocs == 2);
    // many stale sizes do not shut the pool: the last call's block is the one that stays
    for (size_t k = 0; k < 30; k++) {
        Pool::Block held[3];
        for (int i = 0; i < 3; i++) held[i] = p.take((3 + k) * MiB + 7);
        for (int i = 0; i < 3; i++) p.give(held[i]);
        CHECK(g_held <= (long)(64 * MiB));
        const int before = g_allocs;
        const Pool::Block again = p.take((3 + k) * MiB + 7);
        CHECK(g_allocs == before);
        p.give(again);
    }
    // above the budget: never kept
    const int before = g_allocs;
    for (int i = 0; i < 2; i++) p.give(p.take(100 * MiB));
    CHECK(g_allocs == before + 2 && g_held <= (long)(64 * MiB));
    // another device's blocks are not lent
    g_dev = 1;
    const Pool::Block other = p.take(MiB);
    CHECK(g_allocs == before + 3 && other.dev == 1);
    p.give(other);
    g_dev = 0;
    // a failed allocation gives the idle blocks back and tries again; a second failure is reported
    g_fail = 1;
    const Pool::Block big = p.take(200 * MiB);
    CHECK(big.ptr && g_held == (long)(200 * MiB));
    p.give(big);
    g_fail = 2;
    CHECK(!p.take(MiB).ptr);
    p.give(Pool::Block{});
    g_dev = -1;
    CHECK(!p.take(MiB).ptr);
    g_dev = 0;
    std::vector<std::thread> ts;
    for (int t = 0; t < 8; t++)
        ts.emplace_back([&p, t] {
            for (int i = 0; i < 2000; i++) {
                const Pool::Block b = p.take((size_t)(1 + (i * 7 + t) % 20) * 300000);
                *(volatile size_t*)b.ptr = *(size_t*)b.ptr;      // two users of one block: a race
                p.give(b);
            }
        });
    for (std::thread& t : ts) t.join();
    CHECK(g_held <= (long)(64 * MiB));
    CHECK(p.trim() && g_held == 0 && g_live.empty());
    return 0;
}
