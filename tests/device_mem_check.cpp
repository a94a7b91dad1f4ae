// The device memory of the handles (device_mem.cpp) and the pinned blocks and
// staged copies (host_copy.cpp) on the CPU, over a runtime of this file's own:
// device memory is addresses only, so blocks of gibibytes cost nothing, and
// allocations can be made to fail.
//
// Usage: device_mem_check <scenario>; prints "ok" and exits 0 when every check
// of the scenario holds.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <new>
#include <set>
#include <string>
#include <vector>

#include "../include/nido_amd.h"
#include "../nido_amd/csrc/device_mem.h"
#include "../nido_amd/csrc/errors.h"
#include "../nido_amd/csrc/host_copy.h"

static int g_fails = 0;
#define CHECK(c)                                                 \
    do {                                                         \
        if (!(c)) {                                              \
            printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #c);  \
            ++g_fails;                                           \
        }                                                        \
    } while (0)

// ---- the runtime ---------------------------------------------------------------
struct Event {
    int stream = 0;
};
struct Dev {
    size_t capacity = size_t(64) << 30, used = 0, pool_idle = 0, threshold = 0;
    std::map<void*, size_t> live;
    std::vector<size_t> freed_async;      // not yet past a stream synchronisation
    uintptr_t next = 0x100000;
    int oom = 0, frees = 0, bad_frees = 0;
    size_t host_limit = SIZE_MAX;         // larger pinned allocations fail
    int host_allocs = 0, host_frees = 0;
    std::set<int> dead_streams;
} D;
static bool g_throw = false;              // operator new fails

void* operator new(size_t n)
{
    void* p = g_throw ? nullptr : malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

// The runtime's own lists grow all the same.
struct Grow {
    bool was = g_throw;
    Grow() { g_throw = false; }
    ~Grow() { g_throw = was; }
};

// Frees that were waited for go back to the system above the pool's threshold.
static void settle()
{
    for (size_t b : D.freed_async) D.pool_idle += b;
    D.freed_async.clear();
    if (D.pool_idle > D.threshold) D.pool_idle = D.threshold;
}
static size_t held()
{
    size_t n = D.used + D.pool_idle;
    for (size_t b : D.freed_async) n += b;
    return n;
}
static hipError_t alloc(void** p, size_t n)
{
    Grow grow;
    const size_t reuse = std::min(D.pool_idle, n);
    if (held() - reuse + n > D.capacity) {
        ++D.oom;
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    D.pool_idle -= reuse;
    D.used += n;
    *p = reinterpret_cast<void*>(D.next);
    D.next += n;
    D.live[*p] = n;
    return hipSuccess;
}
static hipError_t release_to_pool(void* p, bool async)
{
    Grow grow;
    const auto it = D.live.find(p);
    if (it == D.live.end()) {
        ++D.bad_frees;
        return hipErrorInvalidValue;
    }
    D.used -= it->second;
    if (async) D.freed_async.push_back(it->second);
    D.live.erase(it);
    ++D.frees;
    return hipSuccess;
}
static int id(hipStream_t s) { return (int)reinterpret_cast<uintptr_t>(s); }

extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMemPoolCreate(hipMemPool_t* p, const hipMemPoolProps*)
{
    *p = reinterpret_cast<hipMemPool_t>(&D);
    return hipSuccess;
}
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr a, void* v)
{
    if (a == hipMemPoolAttrReleaseThreshold) D.threshold = (size_t)*static_cast<uint64_t*>(v);
    return hipSuccess;
}
hipError_t hipMemPoolGetAttribute(hipMemPool_t, hipMemPoolAttr a, void* v)
{
    size_t freed = 0;
    for (size_t b : D.freed_async) freed += b;
    uint64_t& x = *static_cast<uint64_t*>(v);
    if (a == hipMemPoolAttrReservedMemCurrent) x = D.used + freed + D.pool_idle;
    else if (a == hipMemPoolAttrUsedMemCurrent) x = D.used;
    else return hipErrorInvalidValue;
    return hipSuccess;
}
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t keep)
{
    D.pool_idle = std::min(D.pool_idle, keep);
    return hipSuccess;
}
hipError_t hipMallocFromPoolAsync(void** p, size_t n, hipMemPool_t, hipStream_t) { return alloc(p, n); }
hipError_t hipFreeAsync(void* p, hipStream_t) { return release_to_pool(p, true); }
hipError_t hipMalloc(void** p, size_t n) { return alloc(p, n); }
hipError_t hipFree(void* p) { return release_to_pool(p, false); }
hipError_t hipStreamSynchronize(hipStream_t)
{
    settle();
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    *p = n <= D.host_limit ? malloc(n) : nullptr;
    D.host_allocs += *p != nullptr;
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p)
{
    ++D.host_frees;
    free(p);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = reinterpret_cast<hipEvent_t>(new Event);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    delete reinterpret_cast<Event*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    reinterpret_cast<Event*>(e)->stream = id(s);
    return hipSuccess;
}
// An event still refers to the stream it was recorded on last.
hipError_t hipEventSynchronize(hipEvent_t e)
{
    return D.dead_streams.count(reinterpret_cast<Event*>(e)->stream) ? hipErrorContextIsDestroyed : hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
}

namespace nido {
int set_error(int code, const char*, ...) { return code; }
}  // namespace nido

using nido::DeviceMem;
static hipStream_t stream(int i) { return reinterpret_cast<hipStream_t>((uintptr_t)i); }
constexpr size_t GiB = size_t(1) << 30, MiB = size_t(1) << 20;

// In the cache alone.
static size_t kept()
{
    const size_t pool = held() - D.used;
    CHECK(DeviceMem::cached() >= pool);
    return DeviceMem::cached() - pool;
}
// held() without what the pool may keep.
static size_t held_here() { return held() - D.pool_idle; }

static void* get(DeviceMem& m, size_t n)
{
    void* p = nullptr;
    CHECK(m.get(&p, n) == hipSuccess && p);
    return p;
}

// What a handle frees is kept, within the stated bounds, for it and for others;
// the rest is back with the system once the stream has been waited for.
static void bounded()
{
    DeviceMem a, b;
    a.open(stream(1));
    b.open(stream(2));
    std::vector<void*> v;
    for (int i = 0; i < 24; ++i) v.push_back(get(i % 2 ? a : b, GiB));
    CHECK(held() == 24 * GiB);
    for (int i = 0; i < 24; ++i) (i % 2 ? a : b).put(v[(size_t)i]);
    // up to kIdleKeep each until the streams are waited for
    CHECK(D.used == 2 * DeviceMem::kIdleKeep);
    settle();
    a.release();
    b.release();
    CHECK(kept() == 4 * GiB);
    CHECK(held_here() == 4 * GiB && D.pool_idle <= DeviceMem::kPoolKeep);
    // more than the cache keeps, handle by handle: the oldest go back
    DeviceMem h[6];
    std::vector<void*> w;
    for (int i = 0; i < 6; ++i) {
        h[i].open(stream(3 + i));
        for (int r = 0; r < 3; ++r) w.push_back(get(h[i], (size_t)(600 + 16 * i) * MiB));
    }
    for (int i = 0; i < 6; ++i) {
        for (int r = 0; r < 3; ++r) h[i].put(w[(size_t)(3 * i + r)]);
        settle();
        h[i].release();
        settle();
        CHECK(kept() <= DeviceMem::kCacheKeep);
        CHECK(held_here() == kept() + (size_t)3 * [&] {
            size_t n = 0;
            for (int k = i + 1; k < 6; ++k) n += D.live.at(w[(size_t)(3 * k)]);
            return n;
        }());
    }
    CHECK(kept() > DeviceMem::kCacheKeep - 3 * GiB / 4);
    // the last ones are still there and are handed out again
    const int frees = D.frees;
    const uintptr_t next = D.next;
    void* p = get(b, 680 * MiB);
    CHECK(std::find(w.begin() + 9, w.end(), p) != w.end());
    CHECK(D.next == next && D.frees == frees);
    b.put(p);
    settle();
    b.release();
    // many small blocks: a bounded number
    v.clear();
    for (size_t i = 0; i < DeviceMem::kCacheBlocks + 500; ++i) v.push_back(get(a, 1024));
    for (void* x : v) a.put(x);
    settle();
    a.release();
    settle();
    CHECK(held_here() == kept() && kept() <= DeviceMem::kCacheKeep);
    CHECK(D.bad_frees == 0);
}

// An allocation that fails is tried again with everything idle given back.
static void retry()
{
    D.capacity = 10 * GiB;
    DeviceMem a, b;
    a.open(stream(1));
    b.open(stream(2));
    void *x = get(a, 3 * GiB / 2), *y = get(a, GiB / 2), *z = get(b, GiB);
    a.put(x);
    a.put(y);
    settle();
    a.release();                       // 2 GiB in the cache
    b.put(z);                          // 1 GiB idle in b
    CHECK(held() == 3 * GiB && kept() == 2 * GiB);
    void* big = get(b, 9 * GiB);
    CHECK(D.oom == 1 && kept() == 0 && held() == 9 * GiB);
    // one that cannot succeed fails, and what is there stays usable
    void* p = big;
    CHECK(b.get(&p, 2 * GiB) == hipErrorOutOfMemory && p == nullptr);
    a.put(get(a, GiB / 2));
    b.put(big);                        // too large to keep
    settle();
    a.release();
    b.release();
    CHECK(kept() == GiB / 2 && held() <= GiB / 2 + DeviceMem::kPoolKeep && D.bad_frees == 0);
}

// Lists that cannot grow lose no block and let no exception out.
static void no_memory()
{
    DeviceMem a;
    a.open(stream(1));
    std::vector<void*> v;
    for (int i = 0; i < 9; ++i) v.push_back(get(a, GiB / 8));
    g_throw = true;
    a.put(v[0]);
    g_throw = false;
    for (int i = 1; i < 9; ++i) a.put(v[(size_t)i]);
    settle();
    g_throw = true;
    a.release();
    g_throw = false;
    settle();
    CHECK(D.live.size() * (GiB / 8) == kept() && held_here() == kept());
    g_throw = true;
    void* p = nullptr;
    const hipError_t e = a.get(&p, 5 * GiB);
    g_throw = false;
    CHECK(e == hipErrorOutOfMemory && p == nullptr);
    settle();
    CHECK(held_here() == kept() && D.bad_frees == 0);
    nido::PinnedBlock b = nido::pinned_get(4 * MiB);
    CHECK(b.p && b.bytes >= 4 * MiB);
    g_throw = true;
    nido::pinned_put(b);
    g_throw = false;
    CHECK(!b.p && D.host_frees + 1 >= D.host_allocs);
}

// Pinned blocks: reused from a quarter of their size up, 1 GiB idle at most.
static void pinned()
{
    nido::PinnedBlock a = nido::pinned_get(8 * MiB);
    char* const p = a.p;
    nido::pinned_put(a);
    CHECK(!a.p);
    nido::PinnedBlock b = nido::pinned_get(2 * MiB), c = nido::pinned_get(2 * MiB);
    CHECK(b.p == p && c.p != p);
    nido::pinned_put(b);
    nido::pinned_put(c);
    nido::PinnedBlock d = nido::pinned_get(MiB);
    CHECK(d.p == c.p || d.bytes == 2 * MiB);          // the smallest that serves
    nido::pinned_put(d);
    nido::PinnedBlock e = nido::pinned_get(MiB / 4);  // none of theirs: they are more than four times as large
    CHECK(e.bytes == MiB / 4);
    nido::pinned_put(e);
    std::vector<nido::PinnedBlock> v;
    for (int i = 0; i < 5; ++i) v.push_back(nido::pinned_get(300 * MiB));
    for (auto& x : v) nido::pinned_put(x);
    CHECK(D.host_allocs - D.host_frees <= 3 + 3);     // three of 300 MiB fit beside the small ones
    D.host_limit = 100 * MiB;
    nido::PinnedBlock f = nido::pinned_get(500 * MiB);
    CHECK(!f.p);
}

// Staged copies wait for events that they recorded themselves: the kept ones
// still name the stream of an earlier copy, which may be gone.
static void staged()
{
    CHECK(nido::set_staging(4096, 4096) == NIDO_OK);
    std::vector<char> src(50000), dst(50000), back(50000);
    for (size_t i = 0; i < src.size(); ++i) src[i] = (char)(i * 7 + i / 251);
    std::vector<int64_t> ids(9001);
    for (size_t i = 0; i < ids.size(); ++i) ids[i] = (int64_t)(i * 37 % 9001);
    for (int s = 1; s <= 6; ++s) {
        std::fill(dst.begin(), dst.end(), 0);
        std::fill(back.begin(), back.end(), 0);
        CHECK(nido::staged_h2d(dst.data(), src.data(), src.size(), stream(s)) == hipSuccess);
        CHECK(nido::staged_d2h(back.data(), dst.data(), src.size(), stream(s)) == hipSuccess);
        CHECK(dst == src && back == src);
        std::vector<int> out(ids.size());
        CHECK(nido::staged_h2d_ids(out.data(), ids.data(), (int64_t)ids.size(), stream(s)) == hipSuccess);
        CHECK(std::equal(ids.begin(), ids.end(), out.begin()));
        D.dead_streams.insert(s);
    }
}

int main(int argc, char** argv)
{
    const std::map<std::string, void (*)()> all = {
        {"bounded", bounded}, {"retry", retry}, {"no_memory", no_memory}, {"pinned", pinned}, {"staged", staged}};
    const auto it = argc > 1 ? all.find(argv[1]) : all.end();
    if (it == all.end()) return 2;
    it->second();
    if (g_fails) return 1;
    printf("ok\n");
    return 0;
}
