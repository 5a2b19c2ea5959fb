// Checks of the device-block cache's policy (ciflow_amd/csrc/block_cache.h) on
// the CPU, with blocks of host memory: reuse, the size limits of a reuse, the
// bound over all caches, age, a source that runs out, blocks given after the
// close, and several threads on several caches.  Built by tests/test_block_cache.py.
#include "../../ciflow_amd/csrc/block_cache.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <thread>

#define CHECK(c)                                                    \
    do {                                                            \
        if (!(c)) {                                                 \
            std::printf("line %d: %s does not hold\n", __LINE__, #c); \
            std::exit(1);                                           \
        }                                                           \
    } while (0)

using namespace cf;

struct HostSource : BlockSource {
    std::mutex mu;
    std::map<void*, size_t> live;
    size_t bytes = 0, room = ~(size_t)0;
    int allocs = 0, unordered = 0, drains = 0;
    void* alloc(size_t b) override {
        std::lock_guard<std::mutex> lk(mu);
        if (bytes + b > room) return nullptr;
        void* p = std::malloc(b);
        live[p] = b;
        bytes += b;
        ++allocs;
        return p;
    }
    void free(void* p) override {
        std::lock_guard<std::mutex> lk(mu);
        CHECK(live.count(p));
        bytes -= live[p];
        live.erase(p);
        std::free(p);
    }
    void free_unordered(void* p) override {
        ++unordered;
        free(p);
    }
    bool short_of = false;
    void drain() override { ++drains; }
    bool scarce() override { return short_of; }
};

int main() {
    {  // reuse, and only of blocks that hardly exceed the request
        BlockBudget bud;
        bud.limit = 1 << 30;
        HostSource src;
        BlockCache c(&src, &bud);
        size_t g1 = 0, g2 = 0;
        void* p = c.take(1000, &g1);
        CHECK(g1 == 1024 && src.allocs == 1);
        c.give(p, g1);
        CHECK(bud.held() == 1024);
        CHECK(c.take(1024, &g2) == p && g2 == 1024 && bud.held() == 0);
        c.give(p, g1);
        CHECK(c.take(512, &g2) == p && g2 == 1024);  // small: up to twice
        c.give(p, g1);
        void* q = c.take(500, &g2);  // 512 wanted, 1024 serves
        CHECK(q == p && g2 == 1024);
        c.give(q, g2);
        q = c.take(256, &g2);
        CHECK(q != p && g2 == 256);  // more than twice
        c.give(q, g2);
        size_t big = 100u << 20;
        p = c.take(big, &g1);
        c.give(p, g1);
        q = c.take(big - (4u << 20), &g2);  // 4% smaller: a block of its own
        CHECK(q != p);
        c.give(q, g2);
        q = c.take(big - (1u << 20), &g2);
        CHECK(q == p && g2 == big);
        c.give(q, g2);
        const size_t held = bud.held();
        CHECK(held > 0 && c.trim() == held);
        CHECK(src.live.empty() && bud.held() == 0 && c.trim() == 0);
    }
    {  // a device short of memory: large blocks are not kept, small ones are
        BlockBudget bud;
        bud.limit = 1 << 30;
        HostSource src;
        src.short_of = true;
        BlockCache c(&src, &bud);
        size_t g, h;
        void *p = c.take(BlockCache::kLarge, &g), *q = c.take(BlockCache::kLarge - 256, &h);
        c.give(p, g);
        c.give(q, h);
        CHECK(!src.live.count(p) && src.live.count(q) && bud.held() == h);
        src.short_of = false;
        p = c.take(BlockCache::kLarge, &g);
        c.give(p, g);
        CHECK(bud.held() == g + h && bud.trim_all() == g + h && src.live.empty());
    }
    {  // the bound: oldest blocks go first, a block over the bound goes at once
        BlockBudget bud;
        bud.limit = 4096;
        HostSource src;
        BlockCache c(&src, &bud);
        void* p[5];
        size_t g[5];
        for (int i = 0; i < 5; ++i) p[i] = c.take(1024, &g[i]);
        for (int i = 0; i < 5; ++i) c.give(p[i], g[i]);
        CHECK(bud.held() == 4096 && src.bytes == 4096 && !src.live.count(p[0]));
        size_t gb;
        void* big = c.take(8192, &gb);
        c.give(big, gb);
        CHECK(src.bytes == 4096);
        // another cache under the same bound keeps nothing past it
        HostSource src2;
        BlockCache c2(&src2, &bud);
        void* o = c2.take(1024, &gb);
        c2.give(o, gb);
        CHECK(src2.bytes == 0 && bud.held() == 4096);
    }
    {  // age
        BlockBudget bud;
        bud.limit = 1 << 30;
        HostSource src;
        BlockCache c(&src, &bud);
        size_t g, h;
        void* p = c.take(1 << 20, &g);
        c.give(p, g);
        for (uint64_t i = 0; i < BlockCache::kKeepTakes + 2; ++i) {
            void* q = c.take(256, &h);
            c.give(q, h);
        }
        CHECK(!src.live.count(p) && bud.held() == 256);
    }
    {  // a source that runs out gets back what every cache holds
        BlockBudget bud;
        bud.limit = 1 << 20;
        HostSource src, other;
        BlockCache c(&src, &bud), d(&other, &bud);
        src.room = 10000;
        size_t g, h;
        void* p = c.take(4096, &g);
        c.give(p, g);
        void* o = d.take(4096, &h);
        d.give(o, h);
        void* q = c.take(8192, &g);
        CHECK(q && bud.held() == 0 && src.drains == 1 && other.drains == 1 && other.bytes == 0);
        CHECK(c.take(8192, &h) == nullptr);
        c.give(q, g);
    }
    {  // blocks given after the close
        BlockBudget bud;
        bud.limit = 1 << 20;
        HostSource src;
        BlockCache c(&src, &bud);
        size_t g, h;
        void *p = c.take(100, &g), *q = c.take(100, &h);
        c.give(q, h);
        c.close();
        CHECK(src.live.size() == 1 && bud.caches.empty());
        c.give(p, g);
        CHECK(src.live.empty() && src.unordered == 1);
    }
    {  // threads: two on one cache, one on another, one that trims everything
        BlockBudget bud;
        bud.limit = 1 << 16;
        HostSource sa, sb;
        BlockCache a(&sa, &bud), b(&sb, &bud);
        auto work = [](BlockCache* c, unsigned seed) {
            std::vector<std::pair<void*, size_t>> mine;
            for (int i = 0; i < 20000; ++i) {
                seed = seed * 1664525u + 1013904223u;
                if (mine.size() < 8 && (seed >> 30) != 0) {
                    size_t g;
                    void* p = c->take(1 + (seed >> 8) % 8000, &g);
                    std::memset(p, (int)seed, g);
                    mine.emplace_back(p, g);
                } else if (!mine.empty()) {
                    c->give(mine.back().first, mine.back().second);
                    mine.pop_back();
                }
            }
            for (auto& m : mine) c->give(m.first, m.second);
        };
        std::thread t1(work, &a, 1u), t2(work, &a, 2u), t3(work, &b, 3u), t4([&] {
            for (int i = 0; i < 200; ++i) bud.trim_all();
        });
        t1.join();
        t2.join();
        t3.join();
        t4.join();
        CHECK(bud.held() == sa.bytes + sb.bytes && bud.held() <= bud.limit);
        a.close();
        b.close();
        CHECK(sa.live.empty() && sb.live.empty() && bud.held() == 0);
    }
    std::printf("all block cache checks passed\n");
    return 0;
}
