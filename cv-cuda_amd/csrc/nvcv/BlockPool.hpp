// Freed blocks of the default allocator, kept for the allocations that follow.
//
// hipFree waits for all of the device's work and hipMalloc maps memory, so a program that makes its outputs anew for
// every batch paid 27 us and a drained device per tensor (16 x 1080p through four allocating operators: 215 us a pass, of
// which the kernels take 28). A block given back here is not waited for: it goes to `waiting`, whatever stream may
// still use it, and becomes `ready` only after a synchronisation of the whole device that began after it was given
// back. That synchronisation is made on the allocating side, when no ready block fits and either kMostWaiting blocks of
// the size wait or half of the pool's limit is waiting or ready: once in 32 allocations of blocks of up to a 64th of the
// limit, by which time most of them are idle, and in as many as fit half of the limit of larger ones (200 MiB under 1 GiB:
// every third).
//
// Bounds: the blocks held and not in use never exceed `limit` (where one more would, others are freed to make room;
// one larger than a quarter of it is not kept); at every synchronisation the blocks that were ready since the one
// before and found no use are freed; when the device is out of memory, or release() is called, all of them are. Safe with
// any number of threads (one lock, not held across the synchronisation) and streams. At the end of the process the blocks
// are left to the runtime, which may be gone by then.
#ifndef NVCVAMD_BLOCKPOOL_HPP
#define NVCVAMD_BLOCKPOOL_HPP

#include <cstdint>
#include <map>
#include <mutex>
#include <unordered_map>
#include <utility>
#include <vector>

namespace nvcvamd {

// Memory of one kind. Source: `static void *alloc(size_t)` (nullptr: no memory), `static void free(void *)`,
// `static int device()` (the calling thread's, an index) and `static bool synchronize()` (all work of that device; false:
// not possible now).
template<class Source>
class BlockPool
{
public:
    explicit BlockPool(int64_t limit)
        : m_limit(limit)
    {
    }

    void *alloc(int64_t size)
    {
        const int     dev     = Source::device();
        const int64_t rounded = RoundUp(size);
        const bool    kept    = rounded <= m_limit / 4;
        if (kept)
        {
            if (void *p = take(dev, rounded))
            {
                return p;
            }
            if (worthSynchronizing(dev, rounded) && recycle(dev))
            {
                if (void *p = take(dev, rounded))
                {
                    return p;
                }
            }
        }
        // what is never kept is not rounded either: a tensor of half the device's memory would ask for an eighth more
        void *p = Source::alloc((size_t)(kept ? rounded : size));
        if (p == nullptr && giveBack(dev))
        {
            p = Source::alloc((size_t)(kept ? rounded : size));
        }
        if (p == nullptr && kept && rounded != size)
        {
            return Source::alloc((size_t)size); // (not remembered, so freed at once)
        }
        if (p != nullptr && kept)
        {
            try
            {
                std::lock_guard<std::mutex> lock(m_mutex);
                m_inUse[p] = {rounded, dev};
            }
            catch (...) // no host memory
            {
                Source::free(p);
                return nullptr;
            }
        }
        return p;
    }

    void free(void *p) noexcept
    {
        std::vector<void *> drop;
        try
        {
            std::lock_guard<std::mutex> lock(m_mutex);
            auto                        it = m_inUse.find(p);
            if (it != m_inUse.end())
            {
                const Block b = it->second;
                m_inUse.erase(it);
                Device &d      = m_devices[b.device];
                size_t &ofSize = d.waitingOfSize[b.size];
                makeRoom(d, b.size, drop);
                d.waiting.push_back({b.size, p});
                ++ofSize;
                d.held += b.size;
                p = nullptr;
            }
        }
        catch (...)
        {
            // no host memory to remember it by
        }
        for (void *q : drop)
        {
            Source::free(q);
        }
        if (p != nullptr)
        {
            Source::free(p); // larger than what is kept, or not from here
        }
    }

    // Frees every block that is not in use, of all devices.
    void release()
    {
        std::vector<void *> drop;
        {
            std::lock_guard<std::mutex> lock(m_mutex);
            for (auto &d : m_devices)
            {
                takeAll(d.second, drop);
            }
        }
        for (void *p : drop)
        {
            Source::free(p);
        }
    }

private:
    static constexpr size_t kMostWaiting = 32;

    struct Block
    {
        int64_t size;
        int     device;
    };

    struct Device
    {
        std::map<int64_t, std::vector<void *>>   ready;
        std::map<int64_t, size_t>                unused;        // per size: blocks ready since the last synchronisation, never taken
        std::vector<std::pair<int64_t, void *>>  waiting;
        std::unordered_map<int64_t, size_t>      waitingOfSize;
        int64_t                                  held = 0;      // bytes of ready and waiting
    };

    // Sizes of eight steps per power of two (at most an eighth more than asked for from 32 KiB on, and whole multiples of 4 KiB
    // below). Sizes that no memory has are left as they are, for the allocation to refuse.
    static int64_t RoundUp(int64_t size)
    {
        if (size >= int64_t(1) << 48)
        {
            return size;
        }
        int64_t step = 4096;
        while (step * 16 <= size)
        {
            step *= 2;
        }
        return size <= step ? step : (size + step - 1) / step * step;
    }

    // Takes out blocks until one of `size` fits under the limit: ready ones first, of other sizes before its own, then those
    // that have waited longest (freeing them waits for the device, as freeing the new one would). The new one stays: the
    // sizes that a program frees now are those it asks for next, and what is left of earlier ones would stay for good
    // if it had no way out but another request for its own size (256, 240, 224 and 208 MiB freed once under a limit of 1 GiB:
    // 104 MiB were allocated and freed anew every time from then on).
    void makeRoom(Device &d, int64_t size, std::vector<void *> &drop)
    {
        if (d.held + size <= m_limit)
        {
            return;
        }
        size_t most = d.waiting.size();
        for (auto &r : d.ready)
        {
            most += r.second.size();
        }
        drop.reserve(most); // (nothing below throws)
        for (int own = 0; own < 2; ++own)
        {
            for (auto &r : d.ready)
            {
                while (d.held + size > m_limit && !r.second.empty() && (r.first == size) == (own == 1))
                {
                    drop.push_back(r.second.front());
                    r.second.erase(r.second.begin());
                    auto unused = d.unused.find(r.first);
                    if (unused != d.unused.end() && unused->second > 0)
                    {
                        --unused->second; // (the front ones)
                    }
                    d.held -= r.first;
                }
            }
        }
        size_t n = 0;
        for (; d.held + size > m_limit && n < d.waiting.size(); ++n)
        {
            drop.push_back(d.waiting[n].second);
            --d.waitingOfSize.find(d.waiting[n].first)->second;
            d.held -= d.waiting[n].first;
        }
        d.waiting.erase(d.waiting.begin(), d.waiting.begin() + n);
    }

    void *take(int dev, int64_t size)
    {
        std::lock_guard<std::mutex> lock(m_mutex);
        Device                     &d  = m_devices[dev];
        auto                        it = d.ready.find(size);
        if (it == d.ready.end() || it->second.empty())
        {
            return nullptr;
        }
        // the last in first out: the most likely to be in the caches
        void *p    = it->second.back();
        m_inUse[p] = {size, dev};
        it->second.pop_back();
        size_t &unused = d.unused[size];
        unused         = unused < it->second.size() ? unused : it->second.size();
        d.held -= size;
        return p;
    }

    bool worthSynchronizing(int dev, int64_t size)
    {
        std::lock_guard<std::mutex> lock(m_mutex);
        Device                     &d  = m_devices[dev];
        auto                        it = d.waitingOfSize.find(size);
        return it != d.waitingOfSize.end() && it->second > 0 && (it->second >= kMostWaiting || d.held >= m_limit / 2);
    }

    // Waiting blocks become ready; ready ones that nothing took since the last time are freed.
    bool recycle(int dev)
    {
        std::vector<std::pair<int64_t, void *>> idle;
        {
            std::lock_guard<std::mutex> lock(m_mutex);
            Device                     &d = m_devices[dev];
            idle.swap(d.waiting);
            d.waitingOfSize.clear();
            for (auto &b : idle)
            {
                d.held -= b.first;
            }
        }
        const bool          done = Source::synchronize();
        std::vector<void *> drop;
        {
            std::lock_guard<std::mutex> lock(m_mutex);
            Device                     &d = m_devices[dev];
            if (!done)
            {
                for (auto &b : idle)
                {
                    d.waiting.push_back(b);
                    ++d.waitingOfSize[b.first];
                    d.held += b.first;
                }
                return false;
            }
            for (auto &r : d.ready)
            {
                // (the first `unused` of the stack were there all the time)
                size_t n = d.unused[r.first];
                n        = n < r.second.size() ? n : r.second.size();
                drop.insert(drop.end(), r.second.begin(), r.second.begin() + n);
                r.second.erase(r.second.begin(), r.second.begin() + n);
                d.held -= (int64_t)n * r.first;
            }
            for (auto &b : idle)
            {
                // (other threads may have given blocks back meanwhile)
                if (d.held + b.first > m_limit)
                {
                    drop.push_back(b.second);
                    continue;
                }
                d.ready[b.first].push_back(b.second);
                d.held += b.first;
            }
            for (auto &r : d.ready)
            {
                d.unused[r.first] = r.second.size();
            }
        }
        for (void *p : drop)
        {
            Source::free(p);
        }
        return true;
    }

    // Takes out every block of the device that is not in use.
    static void takeAll(Device &d, std::vector<void *> &drop)
    {
        for (auto &r : d.ready)
        {
            drop.insert(drop.end(), r.second.begin(), r.second.end());
        }
        for (auto &b : d.waiting)
        {
            drop.push_back(b.second);
        }
        d = {};
    }

    // Frees every block that is not in use; false if there was none. (Freeing waits for the device's work by itself.)
    bool giveBack(int dev)
    {
        std::vector<void *> drop;
        {
            std::lock_guard<std::mutex> lock(m_mutex);
            takeAll(m_devices[dev], drop);
        }
        for (void *p : drop)
        {
            Source::free(p);
        }
        return !drop.empty();
    }

    const int64_t                     m_limit;
    std::mutex                        m_mutex;
    std::map<int, Device>             m_devices;
    std::unordered_map<void *, Block> m_inUse;
};

} // namespace nvcvamd

#endif // NVCVAMD_BLOCKPOOL_HPP
