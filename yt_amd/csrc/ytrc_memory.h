// ytrc_memory.h -- a context's device memory: the budget and the blocks kept
// from one call for the next.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <set>
#include <utility>
#include <vector>

namespace {

// Device memory of dataset pools, batches and staged fields: freed blocks of
// up to KEPT_BLOCK bytes are kept for the next one, KEPT_TOTAL in all.  A
// program that renders frame after frame makes and frees the same blocks, and
// an hipMalloc of 10 MB took up to 0.47 ms, an hipFree 0.07 ms, beside kernels
// of 0.1 to 0.3 ms.  Used with ctx->mu held; a block is put back only when
// nothing on the device uses it any more.
//
// No allocation fails for the sake of kept blocks: where the device has no
// room, every context of it gives its blocks back and the allocation is tried
// again (alloc).
//
// With a budget, what the context holds stays within it: datasets, batches
// and servers (`used`) and the kept blocks together.  Kept blocks never make
// it refuse anything: they are given back first.  They serve only blocks of
// their own size then, since a larger one in place of a smaller would hold
// more than is counted.
struct DeviceMemory {
    static constexpr size_t KEPT_BLOCK = 32u << 20, KEPT_TOTAL = 96u << 20, KEPT_COUNT = 8;
    uint64_t budget = 0;  // 0: none
    uint64_t used = 0;    // bytes of datasets, batches and servers

    DeviceMemory()
    {
        All &all = everyone();
        std::lock_guard<std::mutex> lk(all.mu);
        all.set.insert(this);
    }
    DeviceMemory(const DeviceMemory &) = delete;
    ~DeviceMemory()
    {
        {
            All &all = everyone();
            std::lock_guard<std::mutex> lk(all.mu);
            all.set.erase(this);
        }
        clear();
    }

    // Whether `bytes` more may be used.
    bool fits(uint64_t bytes) const { return budget == 0 || used + bytes <= budget; }
    // What is left of the budget once `bytes` more are used.
    uint64_t left(uint64_t bytes) const
    {
        return budget == 0 ? UINT64_MAX : (used + bytes < budget ? budget - used - bytes : 0);
    }
    // Gives kept blocks back until they fit beside `more` bytes; the longest
    // kept go first: a program's present sizes stay.
    void make_room(uint64_t more)
    {
        std::lock_guard<std::mutex> lk(mu);
        drop_above(left(more));
    }
    // hipMalloc; where the device has no room, once more without any
    // context's kept blocks.
    template <class T>
    static hipError_t alloc(T **p, size_t bytes)
    {
        hipError_t e = hipMalloc((void **)p, bytes);
        if (e != hipErrorOutOfMemory) return e;
        (void)hipGetLastError();
        All &all = everyone();
        std::lock_guard<std::mutex> lk(all.mu);
        all.full = true;  // (a block put back meanwhile is not kept)
        for (DeviceMemory *m : all.set) m->clear();
        e = hipMalloc((void **)p, bytes);
        all.full = false;
        return e;
    }
    // A block of at least `bytes`, one of the `more` bytes that the caller is
    // about to use: the smallest kept one that is no more than twice as large
    // (with a budget: of that size), else a new one.
    hipError_t get(size_t bytes, uint64_t more, char **p, size_t *cap)
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            int at = -1;
            for (int i = 0; i < (int)kept.size(); i++) {
                const size_t c = kept[(size_t)i].second;
                if (c >= bytes && (budget == 0 ? c / 2 <= bytes : c == bytes) &&
                    (at < 0 || c < kept[(size_t)at].second))
                    at = i;
            }
            if (at >= 0) {
                *p = kept[(size_t)at].first;
                *cap = kept[(size_t)at].second;
                held -= *cap;
                kept.erase(kept.begin() + at);
            }
            drop_above(left(more));
            if (at >= 0) return hipSuccess;
        }
        *p = nullptr;
        *cap = bytes;
        return alloc(p, bytes);
    }
    // Gives a block back; its bytes are no longer among `used`.
    void put(char *p, size_t cap)
    {
        if (cap > KEPT_BLOCK) {
            hipFree(p);
            return;
        }
        std::lock_guard<std::mutex> lk(mu);
        if (everyone().full) {
            hipFree(p);
            return;
        }
        while (!kept.empty() && (held + cap > KEPT_TOTAL || kept.size() >= KEPT_COUNT)) drop();
        kept.push_back({p, cap});
        held += cap;
        drop_above(left(0));
    }

  private:
    std::mutex mu;  // of the kept blocks: another context's thread may clear them
    std::vector<std::pair<char *, size_t>> kept;
    size_t held = 0;

    struct All {
        std::mutex mu;
        std::set<DeviceMemory *> set;
        std::atomic<bool> full{false};
    };
    // (never destroyed: a context may outlive static objects)
    static All &everyone()
    {
        static All *all = new All();
        return *all;
    }

    void drop()
    {
        hipFree(kept.front().first);
        held -= kept.front().second;
        kept.erase(kept.begin());
    }
    void drop_above(uint64_t most)
    {
        while (!kept.empty() && held > most) drop();
    }
    void clear()
    {
        std::lock_guard<std::mutex> lk(mu);
        drop_above(0);
    }
};

}  // namespace
