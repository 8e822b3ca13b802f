// Device memory of BLAS builds: a few freed blocks are kept for the next build. A groom that moves
// is rebuilt every frame with the same sizes, and hipMalloc and hipFree of the hundreds of
// megabytes that a build takes cost more than its kernels (hipFree of 256 MB: 0.27 ms; a rebuild
// of 3.2M curves spent 2.6 of 5.2 ms in some 25 of each).
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>

namespace vk {

// Shared by a context and the BLASes built in it, which may outlive it. Safe with several threads
// and streams: a block is handed to one owner at a time and comes back idle.
class MemPool {
public:
    explicit MemPool(int device) : device_(device) {
        std::lock_guard<std::mutex> g(pools().m);
        next_ = pools().first;
        pools().first = this;
    }
    ~MemPool() {
        {
            std::lock_guard<std::mutex> g(pools().m);
            MemPool** p = &pools().first;
            while (*p != this) p = &(*p)->next_;
            *p = next_;
        }
        close();
    }
    MemPool(const MemPool&) = delete;
    MemPool& operator=(const MemPool&) = delete;

    struct Block {
        void* p = nullptr;
        size_t bytes = 0;
    };

    // A block of at least `bytes` bytes on the pool's device (the current one); of the kept blocks
    // the smallest that fits and is at most a quarter larger.
    hipError_t acquire(size_t bytes, Block* out) {
        {
            std::lock_guard<std::mutex> g(m_);
            int best = -1;
            for (int i = 0; i < count_; ++i)
                if (kept_[i].bytes >= bytes && kept_[i].bytes <= bytes + bytes / 4 + kSlack &&
                    (best < 0 || kept_[i].bytes < kept_[best].bytes))
                    best = i;
            if (best >= 0) {
                *out = kept_[best];
                --count_;
                for (int i = best; i < count_; ++i) kept_[i] = kept_[i + 1];
                return hipSuccess;
            }
        }
        out->bytes = bytes;
        const hipError_t e = retry_trimmed([&] { return hipMalloc(&out->p, bytes); });
        if (e != hipSuccess) *out = Block{};
        return e;
    }

    // `alloc()`, an allocation on the current device, and when memory runs out once more after the
    // blocks that the pools of all contexts keep on the device are freed: what is kept for the next
    // build must not fail a call that would have had the memory without the pools.
    template <class F>
    static hipError_t retry_trimmed(F&& alloc) {
        hipError_t e = alloc();
        if (e != hipErrorOutOfMemory) return e;
        (void)hipGetLastError();
        int device = 0;
        (void)hipGetDevice(&device);
        {
            std::lock_guard<std::mutex> g(pools().m);
            for (MemPool* p = pools().first; p; p = p->next_)
                if (p->device_ == device) p->trim();
        }
        return alloc();
    }

    // A fence is a small allocation: an owner of blocks makes one with them and frees it before it
    // gives them back, since freeing waits for the device. (hipDeviceSynchronize would wait too, but
    // it ends a stream capture that is under way in the process, where hipFree does not: a program may
    // destroy what it no longer needs while it, or another of its threads, records a graph.)
    static hipError_t make_fence(void** f) {
        return retry_trimmed([&] { return hipMalloc(f, 256); });
    }
    // Whether the device was waited for. A null fence: no.
    static bool wait(void* fence) { return fence && hipFree(fence) == hipSuccess; }

    // Takes a block back; the blocks kept longest make room for it. Without `idle` the GPU may still
    // be using it: it is freed.
    void release(Block b, bool idle) {
        if (!b.p) return;
        bool keep = idle && b.bytes >= kMinBytes && b.bytes <= kMaxBytes;
        Block old[kMaxBlocks];
        int n = 0;
        if (keep) {
            std::lock_guard<std::mutex> g(m_);
            keep = !closed_;
            if (keep) {
                size_t held = b.bytes;
                for (int i = 0; i < count_; ++i) held += kept_[i].bytes;
                for (; n < count_ && (count_ - n == kMaxBlocks || held > kMaxBytes); ++n) {
                    old[n] = kept_[n];
                    held -= kept_[n].bytes;
                }
                count_ -= n;
                for (int i = 0; i < count_; ++i) kept_[i] = kept_[i + n];
                kept_[count_++] = b;
            }
        }
        for (int i = 0; i < n; ++i) (void)hipFree(old[i].p);
        if (!keep) (void)hipFree(b.p);
    }

    void trim() {
        Block old[kMaxBlocks];
        int n = 0;
        {
            std::lock_guard<std::mutex> g(m_);
            for (; n < count_; ++n) old[n] = kept_[n];
            count_ = 0;
        }
        for (int i = 0; i < n; ++i) (void)hipFree(old[i].p);
    }

    // Frees the kept blocks and keeps no more (the context is gone).
    void close() {
        {
            std::lock_guard<std::mutex> g(m_);
            closed_ = true;
        }
        trim();
    }

private:
    // Smaller blocks are not kept: hipMalloc and hipFree of up to 1 MiB take 0.4 us each. 1 GiB holds
    // the three blocks of a rebuild of up to 3.7M phantom curves (286 bytes a curve: scratch 184,
    // records 76, nodes 26). A larger one allocates its scratch each time (repeated builds of 3.68M
    // curves take 1.90 ms, of 4.0M 2.37, of 16M 8.0): the limit bounds what an idle context holds back
    // from the rest of the program.
    static constexpr size_t kMinBytes = size_t(1) << 20, kMaxBytes = size_t(1) << 30, kSlack = 4096;
    static constexpr int kMaxBlocks = 8;

    struct Pools {
        std::mutex m;
        MemPool* first = nullptr;
    };
    static Pools& pools() {  // the process's pools
        static Pools p;
        return p;
    }

    MemPool* next_ = nullptr;
    std::mutex m_;
    Block kept_[kMaxBlocks];
    int count_ = 0;
    bool closed_ = false;
    const int device_;
};

// hipMalloc for all device memory of the library that is not a pool's.
template <class T>
hipError_t device_malloc(T** p, size_t bytes) {
    return MemPool::retry_trimmed([&] { return hipMalloc(reinterpret_cast<void**>(p), bytes); });
}

}  // namespace vk
