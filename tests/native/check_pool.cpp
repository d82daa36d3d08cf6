// check_pool.cpp -- drives the device memory pool (boundaryvaluediffeq.jl_amd/csrc/dev_pool.h)
// with an allocator of fixed capacity, built under AddressSanitizer / UndefinedBehaviorSanitizer
// by tests/test_dev_pool.py.  Exit status 0 when every request was served as expected and
// everything went back.
#include "../../boundaryvaluediffeq.jl_amd/csrc/dev_pool.h"

#include <cstdint>
#include <cstdio>
#include <map>
#include <thread>
#include <vector>

namespace {

int failures = 0;
void expect(bool ok, const char *what) {
    if (!ok) {
        std::printf("FAILED: %s\n", what);
        ++failures;
    }
}

// addresses without memory behind them
struct Device {
    size_t capacity, used = 0;
    std::map<void *, size_t> live;
    std::mutex mu;
    uintptr_t next = 4096;
    int allocs = 0;
    explicit Device(size_t c) : capacity(c) {}
    void *alloc(size_t n) {
        std::lock_guard<std::mutex> g(mu);
        if (used + n > capacity) return nullptr;
        void *p = (void *)next;
        next += n + 4096;
        used += n;
        live[p] = n;
        ++allocs;
        return p;
    }
    void free(void *p) {
        std::lock_guard<std::mutex> g(mu);
        auto it = live.find(p);
        expect(it != live.end(), "a block is freed once");
        if (it == live.end()) return;
        used -= it->second;
        live.erase(it);
    }
    DevPool::Alloc on_alloc() { return [this](size_t n) { return alloc(n); }; }
    DevPool::Free on_free() { return [this](void *p) { this->free(p); }; }
};

constexpr size_t MiB = (size_t)1 << 20;

}  // namespace

int main() {
    // large blocks: exactly what is asked for, never kept
    for (size_t bytes : {256 * MiB + 256, 257 * MiB, 1000 * MiB, 12345 * MiB + 512}) {
        Device d(bytes);
        DevPool p(d.on_alloc(), d.on_free());
        size_t got = 0;
        void *q = p.take(bytes, got);
        expect(q && got == bytes, "a large block that just fits");
        if (q) p.give(q, got);
        expect(d.used == 0 && p.held() == 0, "a large block is not kept");
    }
    // up to the limit: a step larger at most, and the bytes themselves where the step does not fit
    for (size_t bytes : {(size_t)1, (size_t)256, (size_t)4096, (size_t)4352, 65 * MiB + 256, 255 * MiB, 256 * MiB}) {
        Device roomy(1024 * MiB), tight(bytes);
        size_t got = 0;
        DevPool a(roomy.on_alloc(), roomy.on_free()), b(tight.on_alloc(), tight.on_free());
        void *q = a.take(bytes, got);
        expect(q && got >= bytes && got <= bytes + bytes / 8 + 4096 && got <= DevPool::kMaxBlock, "rounded size");
        if (q) a.give(q, got);
        q = b.take(bytes, got);
        expect(q && got == bytes, "the last bytes of the device");
        if (q) b.give(q, got);
        expect(tight.used == bytes && b.held() == bytes, "kept");
        q = b.take(bytes, got);
        expect(q != nullptr, "and found again, or given back and asked for anew");
        if (q) b.give(q, got);
    }
    {  // held blocks give way to a request that needs their memory
        Device d(300 * MiB);
        DevPool p(d.on_alloc(), d.on_free());
        size_t g1 = 0, g2 = 0, g3 = 0;
        void *a = p.take(100 * MiB, g1), *b = p.take(150 * MiB, g2);
        p.give(a, g1);
        expect(p.held() == g1 && d.used == g1 + g2, "one block held");
        void *c = p.take(140 * MiB, g3);
        expect(c && d.used == g2 + g3 && p.held() == 0, "the held block made room");
        expect(!p.take(50 * MiB, g1), "nothing left");
        p.give(b, g2);
        p.give(c, g3);
        p.close();
        expect(d.used == 0, "closed: everything back");
        a = p.take(8 * MiB, g1);
        p.give(a, g1);
        expect(d.used == 0, "closed: nothing is kept");
    }
    {  // reuse, and the bound on what is held
        Device d(4096 * MiB);
        DevPool p(d.on_alloc(), d.on_free());
        std::vector<std::pair<void *, size_t>> v;
        for (int i = 0; i < 12; ++i) {
            size_t got = 0;
            void *q = p.take(200 * MiB, got);
            v.emplace_back(q, got);
        }
        for (auto &b : v) p.give(b.first, b.second);
        expect(p.held() <= DevPool::kMaxHeld && d.used == p.held() && p.held() >= 800 * MiB, "bounded");
        const int before = d.allocs;
        size_t got = 0;
        void *q = p.take(199 * MiB, got);
        expect(q && d.allocs == before, "reused");
        p.give(q, got);
        q = p.take(100 * MiB, got);
        expect(d.allocs == before + 1 && got < 120 * MiB, "a far larger block is not handed out");
        p.give(q, got);
    }
    {  // threads
        Device d(4096 * MiB);
        DevPool p(d.on_alloc(), d.on_free());
        std::vector<std::thread> th;
        for (int t = 0; t < 4; ++t)
            th.emplace_back([&p, t] {
                for (int i = 0; i < 500; ++i) {
                    size_t got = 0;
                    void *q = p.take((size_t)(1 + (i * 7 + t) % 30) * MiB, got);
                    if (q) p.give(q, got);
                }
            });
        for (auto &t : th) t.join();
        expect(d.used == p.held(), "nothing lost between threads");
        p.release();
        expect(d.used == 0, "released");
    }
    std::printf("%s: %d failures\n", failures ? "FAIL" : "OK", failures);
    return failures ? 1 : 0;
}
