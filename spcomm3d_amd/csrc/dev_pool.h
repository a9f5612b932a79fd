// Device memory of the plans and of the plan builder's scratch, kept between plans.
//
// A program that plans a new pattern every few calls (the reference remaps its indices before
// every group of five, miniapp/bench_both.cpp:196-205) asks for some thirty arrays of the same
// sizes each time, and hipMalloc and hipFree of blocks this large map and unmap memory and wait
// for the device: R-MAT 20, fp64 K = 64, remaps + plan + ten calls + destruction, 25.0 ms with them
// (61 the first time) and 16.0 from a pool, R-MAT 16 7.0 and 2.2.
//
// One pool per context.  Everything that touches a block runs on the context's stream (or is
// joined back to it), so a block can be handed out again at once: what uses it next is queued
// behind what used it last.  Panels and value vectors, whose addresses callers may hand to other
// streams, do not come from here.
//
// Bounded: at most `limit` bytes are kept; beyond that the blocks unused for longest are freed.
// Given back: by trim() (spc3d_host_cache_clear), with the context, and when an allocation of any
// context of the process on the same device fails (trim_all).
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>
#include <new>
#include <unordered_map>
#include <vector>

namespace spc3d {

class DevPool {
  public:
    DevPool() = default;
    DevPool(const DevPool &) = delete;
    DevPool &operator=(const DevPool &) = delete;
    ~DevPool()
    {
        {
            std::lock_guard<std::mutex> lock(registry_mutex());
            for (DevPool **at = &registry(); *at; at = &(*at)->next_)
                if (*at == this) {
                    *at = next_;
                    break;
                }
        }
        trim();
        for (void *p : words_)
            (void)hipHostFree(p);
    }

    // Keeps up to `limit` bytes of `device`'s memory.  Once, before the first block.
    void open(int device, size_t limit)
    {
        device_ = device;
        limit_ = limit;
        std::lock_guard<std::mutex> lock(registry_mutex());
        next_ = registry();
        registry() = this;
    }

    // A block of at least `bytes`; a kept one when it is larger by no more than `spare` (a quarter).
    hipError_t get(void **out, size_t bytes) { return get(out, bytes, bytes / 4); }
    hipError_t get(void **out, size_t bytes, size_t spare)
    {
        *out = nullptr;
        if (bytes == 0)
            return hipSuccess;
        if (bytes > SIZE_MAX - kGrain)
            return hipErrorOutOfMemory;
        bytes = (bytes + kGrain - 1) / kGrain * kGrain;
        try {
            std::lock_guard<std::mutex> lock(mu_);
            auto it = kept_.lower_bound(bytes);
            if (it != kept_.end() && it->first - bytes <= spare) {
                void *p = it->second.p;
                sizes_.emplace(p, it->first);
                kept_bytes_ -= it->first;
                kept_.erase(it);
                *out = p;
                return hipSuccess;
            }
        } catch (const std::bad_alloc &) {
            return hipErrorOutOfMemory;
        }
        void *p = nullptr;
        const hipError_t e = device_alloc(device_, &p, bytes); // (no lock held: it may trim this pool)
        if (e != hipSuccess)
            return e;
        try {
            std::lock_guard<std::mutex> lock(mu_);
            sizes_.emplace(p, bytes);
        } catch (const std::bad_alloc &) {
            (void)hipFree(p);
            return hipErrorOutOfMemory;
        }
        *out = p;
        return hipSuccess;
    }

    // hipMalloc on `device` (which is current), to which every pool's kept blocks there give way.
    static hipError_t device_alloc(int device, void **out, size_t bytes)
    {
        hipError_t e = hipMalloc(out, bytes);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            trim_all(device);
            e = hipMalloc(out, bytes);
        }
        return e;
    }

    // Takes back a block that get() handed out.
    void put(void *p)
    {
        if (!p)
            return;
        std::lock_guard<std::mutex> lock(mu_);
        const auto it = sizes_.find(p);
        const size_t bytes = it == sizes_.end() ? 0 : it->second;
        if (it != sizes_.end())
            sizes_.erase(it);
        if (bytes == 0 || bytes > limit_) {
            (void)hipFree(p);
            return;
        }
        try {
            kept_.emplace(bytes, Kept{p, ++clock_});
        } catch (const std::bad_alloc &) {
            (void)hipFree(p);
            return;
        }
        kept_bytes_ += bytes;
        if (kept_bytes_ > limit_)
            shrink(limit_);
    }

    // A few words of pinned host memory for results on their way down (kWords bytes; null when
    // there is none).  Into pageable memory the runtime stages such a copy and waits twice.
    static constexpr size_t kWords = 1024;
    void *get_words()
    {
        {
            std::lock_guard<std::mutex> lock(mu_);
            if (!words_.empty()) {
                void *p = words_.back();
                words_.pop_back();
                return p;
            }
        }
        void *p = nullptr;
        if (hipHostMalloc(&p, kWords, hipHostMallocDefault) == hipSuccess)
            return p;
        (void)hipGetLastError();
        return nullptr;
    }
    void put_words(void *p)
    {
        if (!p)
            return;
        try {
            std::lock_guard<std::mutex> lock(mu_);
            words_.push_back(p);
        } catch (const std::bad_alloc &) {
            (void)hipHostFree(p);
        }
    }

    // Frees every kept block.
    void trim()
    {
        std::lock_guard<std::mutex> lock(mu_);
        shrink(0);
    }
    // Frees every block that a pool of this process keeps on `device`.
    static void trim_all(int device)
    {
        std::lock_guard<std::mutex> lock(registry_mutex());
        for (DevPool *p = registry(); p; p = p->next_)
            if (p->device_ == device)
                p->trim();
    }

  private:
    struct Kept {
        void *p;
        uint64_t since;
    };
    // Frees kept blocks, the ones unused for longest first, until at most `to` bytes are kept.
    void shrink(size_t to)
    {
        while (kept_bytes_ > to && !kept_.empty()) {
            auto oldest = kept_.begin();
            for (auto it = kept_.begin(); it != kept_.end(); ++it)
                if (it->second.since < oldest->second.since)
                    oldest = it;
            (void)hipFree(oldest->second.p);
            kept_bytes_ -= oldest->first;
            kept_.erase(oldest);
        }
    }
    // The open pools of the process, one after the other.  registry_mutex() is taken before a
    // pool's own and never while one is held.
    static std::mutex &registry_mutex()
    {
        static std::mutex *m = new std::mutex(); // outlives every context, static ones too
        return *m;
    }
    static DevPool *&registry()
    {
        static DevPool *first = nullptr;
        return first;
    }
    DevPool *next_ = nullptr;
    int device_ = 0;
    static constexpr size_t kGrain = 512;
    std::mutex mu_;
    std::vector<void *> words_; // get_words() of as many threads as ever plan at once
    std::multimap<size_t, Kept> kept_; // by size
    std::unordered_map<void *, size_t> sizes_; // of the blocks handed out
    size_t kept_bytes_ = 0, limit_ = 0;
    uint64_t clock_ = 0;
};

// A context's stream and the pool whose blocks are used on it.
struct DevStream {
    hipStream_t st;
    DevPool *pool;
    operator hipStream_t() const { return st; }
};

} // namespace spc3d
