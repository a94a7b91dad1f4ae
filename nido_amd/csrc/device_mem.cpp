// device_mem.cpp -- device memory of the handles (device_mem.h).
#include "device_mem.h"

#include <algorithm>
#include <cstdint>
#include <map>
#include <mutex>

namespace nido {
namespace {

using Block = DeviceMem::Block;

struct Cache {
    std::vector<Block> blocks;   // the oldest first
    size_t bytes = 0;
    hipMemPool_t pool = nullptr;
    bool tried = false;
};
// Never destroyed: handles may outlive static destructors.
std::mutex& g_mu = *new std::mutex;
std::map<int, Cache>& g_cache = *new std::map<int, Cache>;

// Sizes are rounded up to an eighth of their power of two, so that a graph of
// nearly the same size finds the blocks of the one before.
size_t rounded(size_t bytes)
{
    if (bytes <= 512) return 512;
    size_t step = 64;
    while (step * 16 < bytes) step *= 2;
    return (bytes + step - 1) & ~(step - 1);
}

// The smallest block of at least `need` bytes and at most a quarter more.
size_t best_fit(const std::vector<Block>& v, size_t need)
{
    size_t best = v.size();
    for (size_t i = 0; i < v.size(); ++i)
        if (v[i].bytes >= need && v[i].bytes - need <= need / 4 && (best == v.size() || v[i].bytes < v[best].bytes))
            best = i;
    return best;
}

// g_mu is held.
Cache& cache_of(int device)
{
    Cache& c = g_cache[device];
    if (!c.tried) {
        c.tried = true;
        hipMemPoolProps props{};
        props.allocType = hipMemAllocationTypePinned;
        props.handleTypes = hipMemHandleTypeNone;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = device;
        if (hipMemPoolCreate(&c.pool, &props) == hipSuccess) {
            uint64_t keep = DeviceMem::kPoolKeep;
            (void)hipMemPoolSetAttribute(c.pool, hipMemPoolAttrReleaseThreshold, &keep);
        } else {
            (void)hipGetLastError();
            c.pool = nullptr;
        }
    }
    return c;
}

hipMemPool_t pool_of(int device)
{
    std::lock_guard<std::mutex> lk(g_mu);
    return cache_of(device).pool;
}

hipError_t runtime_alloc(void** p, size_t bytes, hipMemPool_t pool, hipStream_t s)
{
    const hipError_t e = pool ? hipMallocFromPoolAsync(p, bytes, pool, s) : hipMalloc(p, bytes);
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
    }
    return e;
}

void runtime_free(void* p, hipMemPool_t pool, hipStream_t s)
{
    if (pool) (void)hipFreeAsync(p, s);
    else (void)hipFree(p);
}

}  // namespace

void DeviceMem::open(hipStream_t s)
{
    s_ = s;
    if (hipGetDevice(&device_) != hipSuccess) device_ = -1;
}

hipError_t DeviceMem::get(void** p, size_t bytes)
{
    *p = nullptr;
    const size_t need = rounded(bytes);
    size_t got = need;
    size_t i = best_fit(idle_, need);
    hipMemPool_t pool = nullptr;
    if (i < idle_.size()) {
        *p = idle_[i].p;
        got = idle_[i].bytes;
        idle_bytes_ -= got;
        idle_.erase(idle_.begin() + (ptrdiff_t)i);
    } else {
        std::lock_guard<std::mutex> lk(g_mu);
        Cache& c = cache_of(device_);
        pool = c.pool;
        i = best_fit(c.blocks, need);
        if (i < c.blocks.size()) {
            *p = c.blocks[i].p;
            got = c.blocks[i].bytes;
            c.bytes -= got;
            c.blocks.erase(c.blocks.begin() + (ptrdiff_t)i);
        }
    }
    hipError_t e = hipSuccess;
    if (!*p) e = runtime_alloc(p, need, pool, s_);
    if (e != hipSuccess) {
        // everything idle goes back, to the system as well
        std::vector<Block> all;
        {
            std::lock_guard<std::mutex> lk(g_mu);
            Cache& c = cache_of(device_);
            all.swap(c.blocks);
            c.bytes = 0;
        }
        for (const Block& b : all) runtime_free(b.p, pool, s_);
        for (const Block& b : idle_) runtime_free(b.p, pool, s_);
        idle_.clear();
        idle_bytes_ = 0;
        (void)hipStreamSynchronize(s_);
        if (pool) (void)hipMemPoolTrimTo(pool, 0);
        e = runtime_alloc(p, need, pool, s_);
    }
    if (e != hipSuccess) return e;
    try {
        live_[*p] = got;
    } catch (...) {
        runtime_free(*p, pool_of(device_), s_);
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    return hipSuccess;
}

void DeviceMem::put(void* p)
{
    if (!p) return;
    const auto it = live_.find(p);
    const size_t bytes = it == live_.end() ? 0 : it->second;
    if (bytes) live_.erase(it);
    if (bytes && idle_bytes_ + bytes <= kIdleKeep) {
        try {
            idle_.push_back(Block{static_cast<char*>(p), bytes});
            idle_bytes_ += bytes;
            return;
        } catch (...) {   // no room for the list: it goes back
        }
    }
    runtime_free(p, pool_of(device_), s_);
}

void DeviceMem::release()
{
    if (idle_.empty()) return;
    std::vector<Block> out;
    hipMemPool_t pool = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        Cache& c = cache_of(device_);
        pool = c.pool;
        try {
            // the oldest make room
            size_t n = 0, left = c.bytes + idle_bytes_;
            while (n < c.blocks.size() && (left > kCacheKeep || c.blocks.size() - n + idle_.size() > kCacheBlocks))
                left -= c.blocks[n++].bytes;
            out.assign(c.blocks.begin(), c.blocks.begin() + (ptrdiff_t)n);
            c.blocks.reserve(c.blocks.size() + idle_.size());
            c.blocks.erase(c.blocks.begin(), c.blocks.begin() + (ptrdiff_t)n);
            c.blocks.insert(c.blocks.end(), idle_.begin(), idle_.end());
            c.bytes = left;
            idle_.clear();
        } catch (...) {
            out.clear();
        }
    }
    for (const Block& b : out) runtime_free(b.p, pool, s_);
    for (const Block& b : idle_) runtime_free(b.p, pool, s_);   // where the cache could not take them
    idle_.clear();
    idle_bytes_ = 0;
}

size_t DeviceMem::cached()
{
    int device = -1;
    if (hipGetDevice(&device) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lk(g_mu);
    const auto it = g_cache.find(device);
    if (it == g_cache.end()) return 0;
    size_t n = it->second.bytes;
    uint64_t reserved = 0, used = 0;
    if (it->second.pool &&
        hipMemPoolGetAttribute(it->second.pool, hipMemPoolAttrReservedMemCurrent, &reserved) == hipSuccess &&
        hipMemPoolGetAttribute(it->second.pool, hipMemPoolAttrUsedMemCurrent, &used) == hipSuccess && reserved > used)
        n += (size_t)(reserved - used);
    return n;
}

}  // namespace nido
