// Device memory of one synchronous call, lent from a few idle blocks: hipMalloc and hipFree
// (which waits for the whole device) cost more than a small call's kernels.
#pragma once

#include <cstddef>
#include <mutex>

namespace gpumpi {

// Memory: static bool device(int*), the calling thread's device; static void* alloc(size_t),
// nullptr on failure; static bool free(void*).
template <class Memory>
class WorkspacePool {
public:
    static constexpr size_t kIdleBlocks = 8, kIdleBytes = 64u << 20;
    struct Block {
        void* ptr = nullptr;
        size_t bytes = 0;
        int dev = -1;
    };

    // Sizes go up in eighths of a power of two from 64 KiB: an eighth at most is lent in vain,
    // and calls of nearly the same size share a block.
    static size_t rounded(size_t need) {
        if (need > kIdleBytes) return need;     // never kept
        if (need <= 65536) return 65536;
        size_t top = 131072;
        while (top < need) top *= 2;
        return (need + top / 16 - 1) / (top / 16) * (top / 16);
    }

    // A block of at least `need` bytes on the calling thread's device: the smallest idle one
    // that is large enough, or new memory (the idle blocks are given back if that fails).
    Block take(size_t need) {
        Block b;
        if (!Memory::device(&b.dev)) return b;
        b.bytes = rounded(need);
        {
            std::lock_guard<std::mutex> g(mu_);
            int best = -1;
            for (int i = 0; i < count_; i++)
                if (idle_[i].dev == b.dev && idle_[i].bytes >= b.bytes && (best < 0 || idle_[i].bytes < idle_[best].bytes))
                    best = i;
            if (best >= 0) return remove(best);
        }
        b.ptr = Memory::alloc(b.bytes);
        if (!b.ptr) {
            trim();
            b.ptr = Memory::alloc(b.bytes);
        }
        return b;
    }

    // Gives a block back whose last use the caller has waited for.  It stays idle, the blocks
    // that have lain idle longest make room for it; a block above the whole budget is freed.
    void give(const Block& b) {
        if (!b.ptr) return;
        Block gone[kIdleBlocks];
        int n = 0;
        const bool keep = b.bytes <= kIdleBytes;
        if (keep) {
            std::lock_guard<std::mutex> g(mu_);
            while (count_ == (int)kIdleBlocks || bytes_ > kIdleBytes - b.bytes) gone[n++] = remove(0);
            idle_[count_++] = b;
            bytes_ += b.bytes;
        }
        for (int i = 0; i < n; i++) Memory::free(gone[i].ptr);
        if (!keep) Memory::free(b.ptr);
    }

    bool trim() {
        Block gone[kIdleBlocks];
        int n = 0;
        {
            std::lock_guard<std::mutex> g(mu_);
            while (count_ > 0) gone[n++] = remove(count_ - 1);
        }
        bool ok = true;
        for (int i = 0; i < n; i++) ok = Memory::free(gone[i].ptr) && ok;
        return ok;
    }

private:
    Block remove(int i) {
        const Block b = idle_[i];
        for (int k = i; k + 1 < count_; k++) idle_[k] = idle_[k + 1];
        count_--;
        bytes_ -= b.bytes;
        return b;
    }

    std::mutex mu_;
    Block idle_[kIdleBlocks];      // the longest idle first
    int count_ = 0;
    size_t bytes_ = 0;
};

}  // namespace gpumpi
