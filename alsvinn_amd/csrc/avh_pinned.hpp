// Pinned host memory of the solvers and batches of a context, in slots:
// allocating a page of it takes 0.1 ms, as long as the rest of a solver.
//
// Solvers and batches hold the pool itself and not their context, so either
// may be destroyed first: the page goes with whoever is last, and what the
// device still writes through a solver's slot stays mapped until that solver
// has waited for it.
#pragma once
#include <cstddef>
#include <memory>
#include <mutex>

namespace avh {

constexpr size_t PINNED_SLOT = 512;
constexpr int PINNED_SLOTS = 64;

class PinnedPool {
public:
    typedef void* (*Allocate)(size_t bytes);  // nullptr if there is none
    typedef void (*Release)(void*);
    PinnedPool(Allocate a, Release r) : allocate(a), release(r) {}
    PinnedPool(const PinnedPool&) = delete;
    PinnedPool& operator=(const PinnedPool&) = delete;
    ~PinnedPool() {
        if (page) release(page);
    }

    // A slot, or an allocation of its own once all are taken; nullptr if there
    // is none.
    void* take() {
        std::lock_guard<std::mutex> g(lock);
        if (!page) page = (char*)allocate(PINNED_SLOT * PINNED_SLOTS);
        for (int i = 0; page && i < PINNED_SLOTS; ++i)
            if (!(used >> i & 1)) {
                used |= 1ull << i;
                return page + i * PINNED_SLOT;
            }
        return allocate(PINNED_SLOT);
    }
    // Whoever gives a slot back has waited for the device's last access.
    void give(void* p) {
        std::lock_guard<std::mutex> g(lock);
        char* const c = (char*)p;
        if (page && c >= page && c < page + PINNED_SLOT * PINNED_SLOTS) used &= ~(1ull << ((c - page) / PINNED_SLOT));
        else release(p);
    }

private:
    Allocate allocate;
    Release release;
    std::mutex lock;
    char* page = nullptr;
    unsigned long long used = 0;  // one bit a slot
};

// One slot, given back when its owner goes.
class PinnedSlot {
public:
    PinnedSlot() = default;
    PinnedSlot(const PinnedSlot&) = delete;
    PinnedSlot& operator=(const PinnedSlot&) = delete;
    ~PinnedSlot() {
        if (at) pool->give(at);
    }
    void* take(const std::shared_ptr<PinnedPool>& from) {
        pool = from;
        return at = pool->take();
    }

private:
    std::shared_ptr<PinnedPool> pool;
    void* at = nullptr;
};

}  // namespace avh
