// dev_pool.h -- blocks of device memory kept between calls.  Plain C++ (the allocator is
// passed in): bvp_internal.h gives it hipMalloc and hipFree, the host checks one of their own.
#pragma once

#include <cstddef>
#include <functional>
#include <map>
#include <mutex>
#include <utility>

// Device blocks of a context that freed arenas leave for later ones (hipMalloc and hipFree
// cost tens of microseconds each, and a call needs a handful of blocks: a lone pendulum solve
// takes 0.46 ms, 0.89 ms with some 35 allocations and 17 small uploads per call).  At most kMaxHeld
// bytes are held, no block above kMaxBlock; the rest, and everything when the context is
// destroyed, goes back to the device.  Work on pooled memory is enqueued on the context's one
// stream, so a block handed on is rewritten only after its last reader; what other streams may
// read is not pooled (networks) or waits for them first (bvp_batch::foreign).
class DevPool {
  public:
    static constexpr size_t kMaxHeld = (size_t)1 << 30, kMaxBlock = (size_t)256 << 20;
    typedef std::function<void *(size_t)> Alloc;  // null when the memory is not there
    typedef std::function<void(void *)> Free;
    DevPool(Alloc alloc, Free free) : alloc_(std::move(alloc)), free_(std::move(free)) {}
    DevPool(const DevPool &) = delete;
    DevPool &operator=(const DevPool &) = delete;
    ~DevPool() { close(); }

    // a block of at least `bytes` (its true size in got), or null
    void *take(size_t bytes, size_t &got) {
        got = bytes;
        if (bytes <= kMaxBlock) {
            // sizes in steps of an eighth of their power of two, so that blocks of nearly the
            // same calls fit each other; larger blocks are never kept and asked for as they are
            size_t step = 4096;
            while (step * 16 < bytes) step *= 2;
            got = (bytes + step - 1) / step * step;
            std::lock_guard<std::mutex> g(mu_);
            auto it = held_.lower_bound(got);
            if (it != held_.end() && it->first <= got + got / 4) {
                void *p = it->second;
                got = it->first;
                held_bytes_ -= got;
                held_.erase(it);
                return p;
            }
        }
        if (void *p = alloc_(got)) return p;
        release();  // the held blocks may be what is missing
        if (void *p = alloc_(got)) return p;
        if (got == bytes) return nullptr;
        got = bytes;  // or the step
        return alloc_(got);
    }

    void give(void *p, size_t bytes) {
        {
            std::lock_guard<std::mutex> g(mu_);
            if (!closed_ && bytes <= kMaxBlock && held_bytes_ + bytes <= kMaxHeld) {
                held_.emplace(bytes, p);
                held_bytes_ += bytes;
                return;
            }
        }
        free_(p);
    }

    // bytes held, free for the next arena
    size_t held() {
        std::lock_guard<std::mutex> g(mu_);
        return held_bytes_;
    }

    // frees the held blocks
    void release() {
        std::multimap<size_t, void *> out;
        {
            std::lock_guard<std::mutex> g(mu_);
            out.swap(held_);
            held_bytes_ = 0;
        }
        for (auto &b : out) free_(b.second);
    }

    // release(), and hold nothing from now on
    void close() {
        {
            std::lock_guard<std::mutex> g(mu_);
            closed_ = true;
        }
        release();
    }

  private:
    Alloc alloc_;
    Free free_;
    std::mutex mu_;
    std::multimap<size_t, void *> held_;
    size_t held_bytes_ = 0;
    bool closed_ = false;
};
