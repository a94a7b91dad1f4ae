// Stands before the HIP runtime in a test's child process and makes chosen
// calls fail on the host, as they would when the runtime is out of something;
// every kernel that is launched runs as usual.  Loaded with RTLD_GLOBAL before
// libnido_amd.so, whose references it then satisfies; shim_init() names the
// runtime that the calls go on to.
#include <dlfcn.h>
#include <stdint.h>
#include <stdlib.h>

#include <hip/hip_runtime_api.h>

#include <map>
#include <mutex>

namespace {
void* g_hip = nullptr;
int g_launch = 0, g_launches = 0;   // g_launches launches from the g_launch-th on fail (0: none)
hipError_t g_last = hipSuccess;
std::mutex g_mu;
std::map<void*, size_t> g_blocks;   // what the pool handed out
size_t g_used = 0, g_limit = 0;     // its sum; beyond g_limit (0: none) allocations fail
size_t g_pinned_max = SIZE_MAX;     // larger pinned allocations fail

template <typename F>
F real(const char* name)
{
    void* p = g_hip ? dlsym(g_hip, name) : nullptr;
    if (!p) abort();
    return reinterpret_cast<F>(p);
}
}  // namespace

extern "C" {
int shim_init(const char* path)
{
    g_hip = dlopen(path, RTLD_NOW | RTLD_NOLOAD);
    return g_hip ? 0 : 1;
}
void shim_fail_launch(int k, int n)
{
    g_launch = k;
    g_launches = n;
}
void shim_pool_limit(size_t bytes) { g_limit = bytes; }
size_t shim_pool_used(void) { return g_used; }
void shim_pinned_max(size_t bytes) { g_pinned_max = bytes; }

hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t s)
{
    if (g_launch > 0 && --g_launch == 0) {
        if (--g_launches > 0) g_launch = 1;
        return g_last = hipErrorLaunchFailure;
    }
    return real<decltype(&hipLaunchKernel)>("hipLaunchKernel")(f, grid, block, args, lds, s);
}

hipError_t hipMallocFromPoolAsync(void** p, size_t n, hipMemPool_t pool, hipStream_t s)
{
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_limit && g_used + n > g_limit) return g_last = hipErrorOutOfMemory;
    const hipError_t e = real<hipError_t (*)(void**, size_t, hipMemPool_t, hipStream_t)>("hipMallocFromPoolAsync")(p, n, pool, s);
    if (e == hipSuccess) g_used += g_blocks[*p] = n;
    return e;
}

hipError_t hipFreeAsync(void* p, hipStream_t s)
{
    std::lock_guard<std::mutex> lk(g_mu);
    const auto it = g_blocks.find(p);
    if (it != g_blocks.end()) {
        g_used -= it->second;
        g_blocks.erase(it);
    }
    return real<decltype(&hipFreeAsync)>("hipFreeAsync")(p, s);
}

hipError_t hipHostMalloc(void** p, size_t n, unsigned flags)
{
    if (n > g_pinned_max) return g_last = hipErrorOutOfMemory;
    return real<hipError_t (*)(void**, size_t, unsigned)>("hipHostMalloc")(p, n, flags);
}

hipError_t hipGetLastError(void)
{
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e != hipSuccess ? e : real<decltype(&hipGetLastError)>("hipGetLastError")();
}
}
