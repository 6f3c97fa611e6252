// The buffer pool's rules over counted host memory; exits non-zero and says
// which check failed.
#include "pool.hpp"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>

using idrs::BufferPool;

static std::atomic<long> g_allocs{0}, g_frees{0}, g_live{0};
static std::atomic<long> g_limit{-1};   // most bytes of live memory (-1: any)

struct Block {
    size_t bytes;
};
static void *get(size_t bytes) {
    if (g_limit >= 0 && g_live + (long)bytes > g_limit) return nullptr;
    g_allocs++;
    g_live += (long)bytes;
    Block *b = (Block *)malloc(sizeof(Block) + 16);
    b->bytes = bytes;
    return b;
}
static void put(void *p) {
    g_frees++;
    g_live -= (long)((Block *)p)->bytes;
    free(p);
}

#define CHECK(c)                                             \
    do {                                                     \
        if (!(c)) {                                          \
            printf("line %d: %s\n", __LINE__, #c);           \
            return 1;                                        \
        }                                                    \
    } while (0)

int main() {
    {   // a size comes back, the one given first first; never more than the cap
        BufferPool p({get, put}, 1000);
        void *a = p.take(100), *b = p.take(100);
        p.give(a, 100);
        p.give(b, 100);
        CHECK(p.take(100) == a && p.take(100) == b && g_allocs == 2);
        p.give(a, 100);
        p.give(b, 100);
        void *big = p.take(1001);
        p.give(big, 1001);
        CHECK(g_frees == 1 && g_live == 200);
        CHECK(p.trim() == 200 && g_live == 0 && p.trim() == 0);
    }
    {   // full of old sizes: a new size is kept all the same, the longest idle go
        BufferPool p({get, put}, 1000);
        void *old[10];
        for (int i = 0; i < 10; i++) old[i] = p.take(100 + i);
        for (int i = 0; i < 9; i++) p.give(old[i], 100 + i);
        const long before = g_allocs;
        for (int call = 0; call < 50; call++) {
            void *q = p.take(333);
            p.give(q, 333);
            CHECK(g_live <= 1000 + 109);
        }
        CHECK(g_allocs == before + 1);
        CHECK(p.take(108) == old[8] && p.take(100) != old[0]);   // 100 .. was dropped
        g_live = 0;
    }
    {   // no memory left: the idle buffers make room, also for memory not kept
        g_limit = 1000;
        BufferPool p({get, put}, 1000);
        void *a = p.take(600);
        p.give(a, 600);
        void *b = p.allocate(700);
        CHECK(b && g_live == 700);
        CHECK(p.take(600) == nullptr);
        put(b);
        a = p.take(600);
        p.give(a, 600);
        CHECK(p.take(601) != nullptr && g_live == 601);
        g_limit = -1;
        g_live = 0;
    }
    {   // threads
        BufferPool p({get, put}, 4000);
        std::thread t[8];
        for (int k = 0; k < 8; k++)
            t[k] = std::thread([&p, k] {
                for (int i = 0; i < 2000; i++) {
                    const size_t n = 100 + 37 * ((i * 7 + k) % 23);
                    void *a = p.take(n), *b = p.take(n);
                    if (a == b || ((Block *)a)->bytes != n || ((Block *)b)->bytes != n) abort();
                    p.give(a, n);
                    p.give(b, n);
                    if (i % 500 == 499) p.trim();
                }
            });
        for (auto &q : t) q.join();
        p.trim();
        CHECK(g_live == 0);
    }
    printf("ok\n");
    return 0;
}
