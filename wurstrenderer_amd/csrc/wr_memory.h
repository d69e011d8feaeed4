// wr_memory.h -- device memory that a device handle keeps between calls.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace wr {

// Device memory that outlives the calls which use it, kept by a device handle.
// A caller takes a block and gives it back when its stream has finished with
// it; blocks are handed to one caller at a time, so streams and threads never
// share one, and at most `keep` free blocks of at most `most` bytes are held.
// Blocks are given back in destructors and at C entry points, so nothing here
// allocates host memory or throws.
struct BlockPool {
    struct Block { void *p = nullptr; size_t bytes = 0; };
    static constexpr int kMostKept = 3;
    const int keep;  // at most kMostKept
    const size_t most;
    const bool close_fit;  // blocks of more than twice the size asked for are not handed out
    std::mutex m;
    Block held[kMostKept];
    int n = 0;
    BlockPool(int keep_, size_t most_, bool close_fit_ = false)
        : keep(keep_ < kMostKept ? keep_ : kMostKept), most(most_), close_fit(close_fit_) {}
    BlockPool(const BlockPool &) = delete;
    BlockPool &operator=(const BlockPool &) = delete;
    ~BlockPool() { trim(); }
    // the smallest free block of at least `bytes`, else a new one
    hipError_t take(size_t bytes, Block *out) {
        {
            std::lock_guard<std::mutex> lock(m);
            int best = -1;
            for (int i = 0; i < n; i++)
                if (held[i].bytes >= bytes && (!close_fit || held[i].bytes / 2 <= bytes) &&
                    (best < 0 || held[i].bytes < held[best].bytes))
                    best = i;
            if (best >= 0) {
                *out = held[best];
                held[best] = held[--n];
                return hipSuccess;
            }
        }
        const hipError_t e = hipMalloc(&out->p, bytes);
        if (e != hipSuccess) out->p = nullptr;
        out->bytes = e == hipSuccess ? bytes : 0;
        return e;
    }
    // bytes of the free blocks
    size_t idle() {
        std::lock_guard<std::mutex> lock(m);
        size_t bytes = 0;
        for (int i = 0; i < n; i++) bytes += held[i].bytes;
        return bytes;
    }
    // gives every free block back to the runtime
    void trim() {
        std::lock_guard<std::mutex> lock(m);
        while (n > 0) (void)hipFree(held[--n].p);
    }
    void give(Block b) {
        if (!b.p) return;
        if (b.bytes <= most) {
            std::lock_guard<std::mutex> lock(m);
            if (n < keep) {
                held[n++] = b;
                return;
            }
            // the smallest goes
            for (int i = 0; i < n; i++)
                if (held[i].bytes < b.bytes) {
                    const Block larger = b;
                    b = held[i];
                    held[i] = larger;
                }
        }
        (void)hipFree(b.p);
    }
};

// The pools of a device handle, and the allocations of everything that belongs to
// it, which get what the pools hold idle before they fail.
struct DeviceMemory {
    BlockPool spills{2, size_t(1) << 30};       // traversal stack spill regions, one per scene
    BlockPool geometry{3, size_t(512) << 20, true};  // nodes (both copies) and triangles of GPU-built scenes
    BlockPool build_memory{1, size_t(1) << 30}; // mesh copies and scratch of BVH builds
    void trim() {
        spills.trim();
        geometry.trim();
        build_memory.trim();
    }
    size_t idle() { return spills.idle() + geometry.idle() + build_memory.idle(); }
    // hipMalloc that frees the pools' idle blocks where memory runs out
    hipError_t alloc(void **p, size_t bytes) {
        hipError_t e = hipMalloc(p, bytes);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            trim();
            e = hipMalloc(p, bytes);
        }
        return e;
    }
    hipError_t take(BlockPool &pool, size_t bytes, BlockPool::Block *b) {
        hipError_t e = pool.take(bytes, b);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            trim();
            e = pool.take(bytes, b);
        }
        return e;
    }
};

}  // namespace wr
