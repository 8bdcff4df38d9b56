// dev_arena.hpp -- the device memory of a roadmap (roadmap_internal.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <initializer_list>
#include <new>
#include <vector>

namespace pump {
namespace rmb {

// The device memory of one roadmap: ranges cut from blocks, given back with
// the roadmap.  Where the sizes that follow are known, reserve() makes a block
// of just that size for them; other requests share blocks of 8, 32 and then
// 64 MiB, and one past kWhole, or one that goes back before the roadmap
// (alloc_whole), is an allocation of its own.  A range is handed out once, so
// that a buffer that grows leaves its old range to the kernels still queued
// on it without a wait.  hipMalloc and hipFree of a buffer of 4 MiB take 78
// and 204 us (of 32 MiB 192 and 250): the 60 buffers of a planned problem of
// 1000 samples took 9 of its 14 ms.  Used by one thread at a time, as the
// roadmap is.
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
        bytes = padded(bytes);
        for (Block &b : blocks)
            if ((b.kind == kReserved || (b.kind == kShared && bytes <= kWhole)) &&
                b.bytes - b.used >= bytes)
                return take(b, bytes);
        if (bytes > kWhole)
            return add(bytes, kOwn);
        // a request may be larger than the next block (the first one, or after
        // a refusal): the block is then cut to it
        if (add(std::max(next, bytes), kShared)) {
            next = next * 4 < kLargest ? next * 4 : kLargest;
            return take(blocks.back(), bytes);
        }
        return add(bytes, kOwn); // no room for another block
    }

    // memory that release() gives back to the device whatever its size
    void *alloc_whole(size_t bytes) { return add(padded(bytes), kOwn); }

    // Room for the next requests, of these sizes in any order, in one block of
    // just their sum.  Without the memory for it each request is on its own.
    void reserve(std::initializer_list<size_t> sizes)
    {
        size_t sum = 0;
        for (size_t n : sizes)
            sum += padded(n ? n : 1);
        (void)add(sum, kReserved);
    }

    static size_t padded(size_t bytes) { return (bytes + kAlign - 1) / kAlign * kAlign; }

    void release(void *p)
    {
        for (size_t i = 0; i < blocks.size(); ++i)
            if (blocks[i].kind == kOwn && blocks[i].p == p) {
                hipFree(p);
                blocks.erase(blocks.begin() + (std::ptrdiff_t)i);
                return;
            }
    }

private:
    enum Kind { kShared, kReserved, kOwn };
    struct Block {
        char *p;
        size_t bytes, used;
        Kind kind;
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

    void *add(size_t bytes, Kind kind)
    {
        void *p = nullptr;
        if (hipMalloc(&p, bytes) != hipSuccess) {
            // the failed attempt leaves its error as the thread's last error:
            // clear it, so that a later launch check does not report it
            (void)hipGetLastError();
            return nullptr;
        }
        try {
            blocks.push_back(Block{static_cast<char *>(p), bytes, 0, kind});
        } catch (const std::bad_alloc &) {
            hipFree(p);
            return nullptr;
        }
        return p;
    }
};

} // namespace rmb
} // namespace pump
