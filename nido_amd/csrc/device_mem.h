// device_mem.h -- device memory of the handles.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <unordered_map>
#include <vector>

namespace nido {

// Device memory of one handle, in the order of its stream: a block it frees is
// handed out again to the same handle at once (what follows on the stream comes
// after what the block was used for).  release(), whenever the handle has waited
// for its stream, gives the idle blocks to a cache of the device that all handles
// and threads take from; their uses are over, so no stream matters any more.
// What live handles have freed is so within the bound of the cache, and within
// reach of another one's failed allocation.
// Below both is a memory pool of the runtime (hipMallocFromPoolAsync), whose
// frees do not wait for the whole device.  It keeps up to kPoolKeep of what is
// freed, gives the rest back to the system, 0.3 to 7 ms at a time, and hands out
// a block again for nearly its own size only.  (Told to keep all, it gave back 10
// of 12 GiB all the same, but without a bound; told to keep nothing, a run of 512
// graphs took 160 ms for 144.)  Whole runs with it alone and with the kept blocks
// above it: planted partition of 1,024 vertices 1.5 -> 1.05 ms, Chung-Lu with
// 300 K vertices 33 -> 27, R-MAT scale 20 76 -> 62, 512 graphs 153 -> 137.
// Bounded: kIdleKeep bytes idle in a handle, kCacheKeep in the device's cache,
// the oldest going back first, kPoolKeep in the pool; when an allocation fails,
// everything idle goes back and it is tried again.
// One thread at a time uses a handle, and so its DeviceMem.
class DeviceMem {
public:
    static constexpr size_t kIdleKeep = size_t(2) << 30, kCacheKeep = size_t(8) << 30, kCacheBlocks = 2048,
                            kPoolKeep = size_t(2) << 30;
    struct Block {
        char* p;
        size_t bytes;
    };
    // of the current device
    void open(hipStream_t s);
    hipError_t get(void** p, size_t bytes);
    void put(void* p);
    void release();
    // Bytes idle in the current device's cache and pool: free for new handles,
    // although the runtime counts them as used.
    static size_t cached();

private:
    hipStream_t s_ = nullptr;
    int device_ = -1;
    std::vector<Block> idle_;
    size_t idle_bytes_ = 0;
    std::unordered_map<void*, size_t> live_;
};

}  // namespace nido
