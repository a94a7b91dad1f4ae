// Stands before the HIP runtime in a test's child process and makes chosen
// calls fail on the host, as they would when the runtime is out of something;
// every kernel that is launched runs as usual.  Loaded with RTLD_GLOBAL before
// libnido_amd.so, whose references it then satisfies; shim_init() names the
// runtime that the calls go on to.
#include <dlfcn.h>
#include <stdint.h>
#include <stdlib.h>

#include <hip/hip_runtime_api.h>

namespace {
void* g_hip = nullptr;
int g_launch = 0;              // the g_launch-th launch from now fails (0: none)
hipError_t g_last = hipSuccess;

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
void shim_fail_launch(int k) { g_launch = k; }

hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t s)
{
    if (g_launch > 0 && --g_launch == 0) return g_last = hipErrorLaunchFailure;
    return real<decltype(&hipLaunchKernel)>("hipLaunchKernel")(f, grid, block, args, lds, s);
}

hipError_t hipGetLastError(void)
{
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e != hipSuccess ? e : real<decltype(&hipGetLastError)>("hipGetLastError")();
}
}
