// Device blocks that the runtime keeps between a free and the next
// allocation (pt_runtime.hip).  Plain C++ over a driver of four calls, so
// that the rules run on the host alone.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <mutex>
#include <unordered_map>
#include <vector>

namespace pt {

// No request above this reaches the driver: nothing that large exists, and
// every size at or below it can be rounded up without leaving size_t.
constexpr size_t kMaxBlockBytes = (size_t)PTRDIFF_MAX;

// The size a request of at most kMaxBlockBytes is rounded up to: a multiple
// of 512 bytes and of a sixteenth to an eighth of itself.
inline size_t block_class(size_t bytes)
{
    size_t step = 512;
    while (step <= bytes / 16) step *= 2;
    return (bytes + step - 1) / step * step;
}

// Blocks freed on the home stream (the runtime stream), kept for the next
// allocations there.  A block that is allocated, used and freed in one
// stream's order can go to that stream's next user without a marker on the
// GPU or a call into the driver; hipMallocAsync and hipFreeAsync cost 4-5 us
// of host time each and leave gaps between the kernels around them (an eager
// add of 64 x 64 took 17.5 us, 6 of them its launch; softmax and layerNorm of
// [8192, 4096] fp32 took 102 us with kernels of 87).
//  * Only blocks that were allocated and are freed on the home stream while
//    it is not being captured are kept; every other call goes to the
//    driver's pool as it is.  Any thread may free or take one: whatever a
//    thread queues after taking a block follows what was queued before the
//    free on the same stream.
//  * Sizes are rounded up by block_class, and a block serves its own rounded
//    size only.
//  * At most kKeepBytes are kept; a free that would pass it gives every kept
//    block back first.  They are also given back when an allocation fails, on
//    whatever stream, and the allocation is then tried once more.
//  * The driver's pool holds on to freed memory as long as no more than its
//    threshold is reserved, kept blocks and blocks in use among them.  The
//    same threshold, where one is set (set_threshold), bounds the home
//    stream's blocks here: while those in use and those kept come to more,
//    none are kept.
template <typename Driver>
class KeptBlocks {
public:
    using Stream = typename Driver::Stream;
    using Status = typename Driver::Status;
    static constexpr size_t kKeepBytes = (size_t)8 << 30;

    explicit KeptBlocks(Driver d = Driver()) : driver(d) {}

    Status alloc(void **ptr, size_t size, Stream stream, Stream home)
    {
        if (size > kMaxBlockBytes) return Driver::kNoMemory;
        if (stream == home && !driver.capturing(stream)) {
            const size_t rounded = block_class(size);
            std::lock_guard<std::mutex> lock(mu);
            auto it = kept.find(rounded);
            if (it != kept.end() && !it->second.empty()) {
                *ptr = it->second.back();
                it->second.pop_back();
                bytes -= rounded;
                blocks--;
                live[*ptr] = rounded;
                used += rounded;
                return Driver::kOk;
            }
            const Status st = driver.alloc(ptr, rounded, stream);
            if (st == Driver::kOk) {
                live[*ptr] = rounded;
                used += rounded;
                if (bytes && !fits(bytes)) give_back(home);
                return st;
            }
            // out of memory: without the kept blocks, and without the rounding
            give_back(home);
            driver.synchronize(home);
            return driver.alloc(ptr, size, stream);
        }
        Status st = driver.alloc(ptr, size, stream);
        if (st == Driver::kNoMemory && !driver.capturing(stream) && !driver.capturing(home)) {
            {
                std::lock_guard<std::mutex> lock(mu);
                give_back(home);
            }
            driver.synchronize(home);
            st = driver.alloc(ptr, size, stream);
        }
        return st;
    }

    Status release(void *ptr, Stream stream, Stream home)
    {
        {
            std::lock_guard<std::mutex> lock(mu);
            auto it = live.find(ptr);
            if (it != live.end()) {
                const size_t size = it->second;
                live.erase(it);
                used -= size;
                if (stream == home && fits(size) && !driver.capturing(stream)) {
                    if (!fits(bytes + size)) give_back(home);
                    kept[size].push_back(ptr);
                    bytes += size;
                    blocks++;
                    return Driver::kOk;
                }
            }
        }
        return driver.free(ptr, stream);
    }

    // 0: none
    void set_threshold(size_t most, Stream home)
    {
        std::lock_guard<std::mutex> lock(mu);
        threshold = most ? most : SIZE_MAX;
        if (bytes && !fits(bytes) && !driver.capturing(home)) give_back(home);
    }

    void usage(size_t *kept_bytes, size_t *kept_count)
    {
        std::lock_guard<std::mutex> lock(mu);
        if (kept_bytes) *kept_bytes = bytes;
        if (kept_count) *kept_count = blocks;
    }

private:
    // so many kept bytes, beside the blocks in use
    bool fits(size_t n) const { return n <= kKeepBytes && used <= threshold && n <= threshold - used; }

    // Every kept block back to the driver's pool (the caller holds the lock
    // and the home stream is not being captured).
    void give_back(Stream home)
    {
        for (auto &c : kept)
            for (void *p : c.second) (void)driver.free(p, home);
        kept.clear();
        bytes = blocks = 0;
    }

    Driver driver;
    std::mutex mu;
    std::unordered_map<void *, size_t> live;               // rounded size of blocks handed out
    std::unordered_map<size_t, std::vector<void *>> kept;  // free blocks by rounded size
    size_t used = 0, bytes = 0, blocks = 0, threshold = SIZE_MAX;
};

}  // namespace pt
