// dev_arena.hpp -- the device memory of a roadmap (roadmap_internal.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <new>
#include <vector>

namespace pump {
namespace rmb {

// The device memory of one roadmap: ranges cut from blocks of 8, 32 and then
// 64 MiB, given back with the roadmap; a request past kWhole is an allocation
// of its own and goes back when it is released.  A range is handed out once,
// so that a buffer that grows leaves its old range to the kernels still
// queued on it without a wait.  hipMalloc and hipFree of a buffer of 4 MiB
// take 78 and 204 us (of 32 MiB 192 and 250): the 60 buffers of a planned
// problem of 1000 samples took 9 of its 14 ms.  Used by one thread at a time,
// as the roadmap is.
class DevArena {
public:
    DevArena() = default;
    DevArena(const DevArena &) = delete;
    DevArena &operator=(const DevArena &) = delete;
    ~DevArena()
    {
        for (const Block &b : blocks)
            hipFree(b.p);
    }

    // nullptr when the device (or the host) is out of memory
    void *alloc(size_t bytes)
    {
        bytes = (bytes + kAlign - 1) / kAlign * kAlign;
        if (bytes > kWhole)
            return add(bytes, true);
        for (Block &b : blocks)
            if (!b.whole && b.bytes - b.used >= bytes)
                return take(b, bytes);
        // a request may be larger than the next block (the first one, or after
        // a refusal): the block is then cut to it
        if (add(std::max(next, bytes), false)) {
            next = next * 4 < kLargest ? next * 4 : kLargest;
            return take(blocks.back(), bytes);
        }
        return add(bytes, true); // no room for another block
    }

    void release(void *p)
    {
        for (size_t i = 0; i < blocks.size(); ++i)
            if (blocks[i].whole && blocks[i].p == p) {
                hipFree(p);
                blocks.erase(blocks.begin() + (std::ptrdiff_t)i);
                return;
            }
    }

private:
    struct Block {
        char *p;
        size_t bytes, used;
        bool whole;
    };
    static constexpr size_t kAlign = 256, kWhole = (size_t)16 << 20, kLargest = (size_t)64 << 20;
    std::vector<Block> blocks;
    size_t next = (size_t)8 << 20;

    static void *take(Block &b, size_t bytes)
    {
        void *p = b.p + b.used;
        b.used += bytes;
        return p;
    }

    void *add(size_t bytes, bool whole)
    {
        void *p = nullptr;
        if (hipMalloc(&p, bytes) != hipSuccess) {
            // the failed attempt leaves its error as the thread's last error:
            // clear it, so that a later launch check does not report it
            (void)hipGetLastError();
            return nullptr;
        }
        try {
            blocks.push_back(Block{static_cast<char *>(p), bytes, 0, whole});
        } catch (const std::bad_alloc &) {
            hipFree(p);
            return nullptr;
        }
        return p;
    }
};

} // namespace rmb
} // namespace pump
