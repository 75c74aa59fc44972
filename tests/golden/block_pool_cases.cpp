// BlockPool with a counting stand-in for the device: what it reuses, when it synchronises, what it bounds and gives back.
#include "BlockPool.hpp"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <thread>

using nvcvamd::BlockPool;

static std::atomic<int64_t> g_allocs{0}, g_frees{0}, g_syncs{0};
static std::atomic<int64_t> g_asked{0}, g_most{INT64_MAX}; // bytes of the last request; the largest request there is memory for
static std::atomic<bool>    g_full{false}, g_busy{false};

struct Counting
{
    static void *alloc(size_t size)
    {
        g_asked = (int64_t)size;
        if ((g_full && g_allocs - g_frees > 0) || (int64_t)size > g_most)
        {
            return nullptr;
        }
        // (more than any device has: a sanitizer's malloc would end the program for it)
        if (size >= size_t(1) << 40)
        {
            return nullptr;
        }
        ++g_allocs;
        return std::malloc(size < 65536 ? size : 65536); // (larger ones are not written)
    }
    static void free(void *p)
    {
        ++g_frees;
        std::free(p);
    }
    static int device()
    {
        return 0;
    }
    static bool synchronize()
    {
        ++g_syncs;
        return !g_busy;
    }
};

#define REQUIRE(c)                                                                          \
    do                                                                                      \
    {                                                                                       \
        if (!(c))                                                                           \
        {                                                                                   \
            std::printf("line %d: %s\n", __LINE__, #c);                                     \
            return 1;                                                                       \
        }                                                                                   \
    } while (0)

static void Reset()
{
    g_allocs = g_frees = g_syncs = 0;
    g_full = g_busy = false;
    g_most          = INT64_MAX;
}

int main()
{
    {
        // a block given back is not handed out before a synchronisation that began after it was given back
        Reset();
        BlockPool<Counting> pool(1 << 20);
        std::set<void *>    seen;
        for (int i = 0; i < 32; ++i)
        {
            void *p = pool.alloc(5000);
            REQUIRE(p != nullptr && seen.insert(p).second);
            pool.free(p);
        }
        REQUIRE(g_allocs == 32 && g_syncs == 0);
        void *q = pool.alloc(4097); // the 33rd: synchronises and reuses (sizes are rounded up)
        REQUIRE(g_syncs == 1 && g_allocs == 32 && seen.count(q) == 1);
        for (int i = 0; i < 31; ++i)
        {
            REQUIRE(seen.count(pool.alloc(5000)) == 1);
        }
        REQUIRE(g_allocs == 32 && g_syncs == 1);
        REQUIRE(seen.count(pool.alloc(5000)) == 0 && g_allocs == 33); // nothing waits: no synchronisation
    }
    {
        // half of the limit waiting: fewer blocks suffice; larger than a quarter of the limit: never kept
        Reset();
        BlockPool<Counting> pool(1 << 20);
        for (int i = 0; i < 2; ++i)
        {
            pool.free(pool.alloc(1 << 18));
        }
        REQUIRE(g_allocs == 2 && g_frees == 0);
        void *p = pool.alloc(1 << 18);
        REQUIRE(g_syncs == 1 && g_allocs == 2);
        pool.free(p);
        pool.free(pool.alloc((1 << 18) + 1));
        REQUIRE(g_frees == 1);
        // what is held never exceeds the limit
        void *many[12];
        for (auto &m : many)
        {
            m = pool.alloc(1 << 17);
        }
        const int64_t before = g_frees;
        for (auto &m : many)
        {
            pool.free(m);
        }
        // 8 x 128 KiB are 1 MiB: the 2 x 256 KiB held already and the 4 of them that waited longest make room
        REQUIRE(g_frees - before == 2 + 4);
    }
    {
        // blocks that find no use between two synchronisations are freed; a device that cannot be synchronised now
        Reset();
        BlockPool<Counting> pool(1 << 24);
        void               *a[40];
        for (auto &p : a)
        {
            p = pool.alloc(8192);
        }
        for (auto &p : a)
        {
            pool.free(p);
        }
        g_busy = true;
        void *x = pool.alloc(8192);
        REQUIRE(g_syncs == 1 && g_allocs == 41);
        g_busy = false;
        void *y = pool.alloc(8192);
        REQUIRE(g_syncs == 2 && g_allocs == 41); // 40 are ready, one of them taken
        void *b[33];
        for (auto &p : b)
        {
            p = pool.alloc(65536);
        }
        for (auto &p : b)
        {
            pool.free(p);
        }
        REQUIRE(g_frees == 0);
        void *z = pool.alloc(65536); // the next synchronisation: the 39 that nothing took go
        REQUIRE(g_syncs == 3 && g_frees == 39);
        pool.free(x), pool.free(y), pool.free(z);
        // out of memory: everything not in use is given back and the allocation tried again
        g_full = true;
        void *w = pool.alloc(1 << 16 | 1);
        REQUIRE(w != nullptr && g_allocs - g_frees == 1);
        pool.free(std::malloc(16)); // not from here: passed on
    }
    {
        // sizes that nothing asks for any more do not keep others out
        Reset();
        BlockPool<Counting> pool(1 << 30);
        for (int64_t mib : {256, 240, 224, 208})
        {
            pool.free(pool.alloc(mib << 20));
        }
        for (int i = 0; i < 1000; ++i)
        {
            pool.free(pool.alloc(104 << 20));
        }
        REQUIRE(g_allocs <= 4 + 6 && g_syncs > 0); // (half of the limit holds 5 x 104 MiB)
        REQUIRE(g_frees >= 4);                     // and the others are gone
    }
    {
        // everything kept is given back when asked for, ready and waiting; what is in use is not
        Reset();
        BlockPool<Counting> pool(1 << 20);
        void               *a[40];
        for (auto &p : a)
        {
            p = pool.alloc(5000);
        }
        for (auto &p : a)
        {
            pool.free(p);
        }
        int *used = static_cast<int *>(pool.alloc(5000)); // 39 are ready
        for (int i = 0; i < 3; ++i)
        {
            pool.free(pool.alloc(70000 + 20000 * i)); // others wait
        }
        pool.release();
        REQUIRE(g_allocs - g_frees == 1);
        *used = 1;
        pool.free(used);
        pool.release();
        pool.release();
        REQUIRE(g_allocs == g_frees);
        REQUIRE(pool.alloc(5000) != nullptr);
    }
    {
        // sizes that no memory has are refused
        Reset();
        BlockPool<Counting> pool(1 << 20);
        for (int bits = 50; bits < 64; ++bits)
        {
            volatile int64_t size = (int64_t)((uint64_t(1) << bits) - 1);
            REQUIRE(pool.alloc(size) == nullptr);
        }
    }
    {
        // what is never kept is asked for as it is; what is kept too, where there is no memory for the rounded size
        Reset();
        BlockPool<Counting> pool(1 << 20);
        for (int64_t size : {(int64_t(1) << 18) + 1, (int64_t(1) << 32) + 1, int64_t(0x123456789)})
        {
            void *p = pool.alloc(size);
            REQUIRE(p != nullptr && g_asked == size);
            pool.free(p);
        }
        g_most  = 70000;
        void *p = pool.alloc(70000), *q = pool.alloc(70001);
        REQUIRE(p != nullptr && g_asked == 70001 && q == nullptr);
        pool.free(p);
        REQUIRE(g_allocs == 4 && g_frees == 4);
    }
    {
        // threads
        Reset();
        BlockPool<Counting>      pool(1 << 22);
        std::vector<std::thread> threads;
        std::atomic<int>         wrong{0};
        for (int t = 0; t < 8; ++t)
        {
            threads.emplace_back(
                [&, t]
                {
                    for (int i = 0; i < 4000; ++i)
                    {
                        int *p = static_cast<int *>(pool.alloc(4096 << (i % 5)));
                        *p     = t * 4000 + i;
                        std::this_thread::yield();
                        wrong += *p != t * 4000 + i;
                        pool.free(p);
                    }
                });
        }
        for (auto &t : threads)
        {
            t.join();
        }
        REQUIRE(wrong == 0 && g_allocs < 32000 && g_syncs > 0);
    }
    std::puts("ok");
    return 0;
}
