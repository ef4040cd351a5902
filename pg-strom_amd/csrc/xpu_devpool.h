/*
 * xpu_devpool.h - device buffers of closed sessions, kept for the next ones.
 *
 * A backend opens a session per query, and giving its buffers (a 1 GiB
 * kds_final and its overflow table among them) back to the driver makes the
 * next allocation of that size wait until the driver has cleared the freed
 * memory (a 2M-row star query opened and closed in a row: 42 ms a query,
 * 1.3 ms with the buffers kept).
 *
 * Buffers are reused by device and size, a buffer up to a quarter larger than
 * asked for among them.  At most XPU_POOL_BYTES and XPU_POOL_COUNT stay idle:
 * the ones idle for the longest go back to the driver to make room, so the
 * sizes that are in use stay, whatever was closed before them.  All go back
 * when an allocation fails, pooled or direct, and at xpuhip_shutdown.  A
 * buffer is given back only after the work that used it has completed.
 *
 * Mem is the device's memory: alloc, release, device and OUT_OF_MEMORY.
 */
#ifndef XPU_DEVPOOL_H
#define XPU_DEVPOOL_H

#include <stddef.h>

#include <iterator>
#include <list>
#include <map>
#include <mutex>
#include <utility>

#define XPU_POOL_BYTES      (8ULL << 30)
#define XPU_POOL_COUNT      1024

template <class Mem>
struct DevPool
{
    typedef typename Mem::Error Error;
    typedef std::pair<int, size_t> Key;             /* device, size of the buffer */
    typedef std::list<std::pair<Key, void *>> Ages;

    std::mutex  lock;
    std::mutex  trim_lock;      /* held until everything a trim took is released */
    std::map<void *, Key> live;
    Ages        ages;                               /* idle buffers, oldest first */
    std::multimap<Key, typename Ages::iterator> idle;
    size_t      idle_bytes = 0;

    /* an eighth more than asked for at most, and at least 256 bytes */
    static size_t
    round_up(size_t n)
    {
        size_t step = 256;
        while (step * 16 <= n)
            step <<= 1;
        return n ? (n + step - 1) & ~(step - 1) : step;
    }

    /* a buffer outside the pool (its owner frees it), for which the idle ones
     * make room where the device has none */
    Error
    alloc_direct(void **p, size_t n)
    {
        Error rc = Mem::alloc(p, n);
        if (rc == Mem::OUT_OF_MEMORY)
        {
            trim();
            rc = Mem::alloc(p, n);
        }
        return rc;
    }

    Error
    alloc(void **p, size_t n)
    {
        const size_t sz = round_up(n);
        const Key key(Mem::device(), sz);
        {
            std::lock_guard<std::mutex> g(lock);
            auto it = idle.lower_bound(key);
            if (it != idle.end() && it->first.first == key.first && it->first.second <= sz + sz / 4)
            {
                *p = take(it);
                return Error();
            }
        }
        const Error rc = alloc_direct(p, sz);
        if (rc == Error())
        {
            std::lock_guard<std::mutex> g(lock);
            live[*p] = key;
        }
        return rc;
    }

    void
    free(void *p)
    {
        if (!p)
            return;
        Ages gone;
        {
            std::lock_guard<std::mutex> g(lock);
            auto it = live.find(p);
            if (it == live.end())
                gone.emplace_back(Key(), p);
            else
            {
                const Key key = it->second;
                live.erase(it);
                if (key.second > XPU_POOL_BYTES)
                    gone.emplace_back(key, p);
                else
                {
                    while (idle_bytes + key.second > XPU_POOL_BYTES || ages.size() >= XPU_POOL_COUNT)
                        evict(gone);
                    ages.emplace_back(key, p);
                    idle.emplace(key, std::prev(ages.end()));
                    idle_bytes += key.second;
                }
            }
        }
        for (auto &e : gone)
            Mem::release(e.second);
    }

    void
    trim()
    {
        std::lock_guard<std::mutex> t(trim_lock);
        Ages gone;
        {
            std::lock_guard<std::mutex> g(lock);
            gone.swap(ages);
            idle.clear();
            idle_bytes = 0;
        }
        for (auto &e : gone)
            Mem::release(e.second);
    }

  private:
    /* an idle buffer for use (lock held) */
    void *
    take(typename std::multimap<Key, typename Ages::iterator>::iterator it)
    {
        void *p = it->second->second;
        live[p] = it->first;
        idle_bytes -= it->first.second;
        ages.erase(it->second);
        idle.erase(it);
        return p;
    }
    /* moves the buffer idle for the longest to gone (lock held) */
    void
    evict(Ages &gone)
    {
        const auto old = ages.begin();
        auto it = idle.lower_bound(old->first);
        while (it->second != old)
            ++it;
        idle_bytes -= old->first.second;
        idle.erase(it);
        gone.splice(gone.end(), ages, old);
    }
};

#endif  /* XPU_DEVPOOL_H */
