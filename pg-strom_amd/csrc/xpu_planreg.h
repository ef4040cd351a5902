/*
 * xpu_planreg.h - what the sessions of one plan shape share, by the shape's
 * bytes.
 *
 * Queries that differ in a constant differ in shape, so a process meets any
 * number of them: an entry stays while a session holds it, and of the others
 * the XPU_PLAN_KEEP used last (a shape that comes back after that finds its
 * kernels in the code cache again).
 */
#ifndef XPU_PLANREG_H
#define XPU_PLANREG_H

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#define XPU_PLAN_KEEP       1024

template <class T>
class PlanRegistry
{
    struct Entry
    {
        std::shared_ptr<T> value;
        uint64_t        used = 0;       /* turn of the last get */
    };
    std::mutex      lock;
    std::map<std::string, Entry> shapes;
    uint64_t        turn = 0;
    size_t          sweep_at = 2 * XPU_PLAN_KEEP;

    /* drops all but the XPU_PLAN_KEEP entries used last among those no
     * session holds (lock held: no new holder can appear) */
    void
    sweep()
    {
        std::vector<std::pair<uint64_t, typename std::map<std::string, Entry>::iterator>> old;
        for (auto it = shapes.begin(); it != shapes.end(); ++it)
            if (it->second.value.use_count() == 1)
                old.emplace_back(it->second.used, it);
        if (old.size() > XPU_PLAN_KEEP)
        {
            std::sort(old.begin(), old.end(),
                      [](const auto &a, const auto &b) { return a.first < b.first; });
            for (size_t i = 0; i < old.size() - XPU_PLAN_KEEP; i++)
                shapes.erase(old[i].second);
        }
        /* a sweep for every XPU_PLAN_KEEP new shapes */
        sweep_at = shapes.size() + XPU_PLAN_KEEP;
    }

  public:
    std::shared_ptr<T>
    get(const std::string &key)
    {
        std::lock_guard<std::mutex> g(lock);
        auto it = shapes.find(key);
        if (it == shapes.end())
        {
            if (shapes.size() >= sweep_at)
                sweep();
            it = shapes.emplace(key, Entry()).first;
            it->second.value = std::make_shared<T>();
        }
        it->second.used = ++turn;
        return it->second.value;
    }
    size_t
    size()
    {
        std::lock_guard<std::mutex> g(lock);
        return shapes.size();
    }
};

#endif  /* XPU_PLANREG_H */
