// noalloc.hip -- modularity of a caller-supplied partition without any
// device allocation.
//
// nido_compute_modularity evaluates Q for the partition a handle holds; the
// handle owns its state and its reduction buffers, all allocated when it was
// created.  Callers that cannot allocate device memory at all -- code under
// HIP graph capture, tight serving loops, harnesses that forbid hipMalloc --
// cannot create a handle.  nido_modularity_noalloc takes the CSR and the
// community of every vertex as device arrays and computes the same Q (the
// same exact Q64.64 sums, rounded once, so the same bits) with its working
// memory in one file-scope device array.  That array is sized for
// kNoAllocMaxVertices communities; every GPU the library runs on holds it
// until the process ends.
//
// The array's name is a host-side stand-in for the symbol, not a device
// address: the first call on a device, with that device current, resolves
// it with hipGetSymbolAddress and keeps the address per device; every kernel
// argument and fill after that uses the kept address.
//
// Calls on one GPU share its array: each call clears what it sums into
// before using it (with a fill kernel, never hipMemsetAsync, so the launches
// can be captured into a graph; the flag of bad input, which that same
// kernel may set, is cleared by the last kernel of the call, and by an extra one
// where a launch of the call failed), and two calls whose launches overlap on
// one GPU -- on different streams without ordering between them -- race on it.
#include <atomic>
#include <mutex>

#include "../../include/nido_amd.h"
#include "device_common.h"
#include "errors.h"

using namespace nido;

namespace {

constexpr int64_t kNoAllocMaxVertices = NIDO_NOALLOC_MAX_VERTICES;
// [0, max) community totals a_c, then three partial sums per workgroup
// (internal weight, 2m, square terms), then a flag set when an id lies outside
// [0, nv).  Workgroups leave partials instead of adding to one sum: an atomic
// on one address takes its turn at the memory side, about 100 ns each for the
// whole GPU, which was most of the time here.
constexpr int kNoAllocBlocks = 2048;
constexpr int64_t kScratchFx = kNoAllocMaxVertices + 3 * kNoAllocBlocks + 1;

__device__ __align__(256) fx_t scratch[kScratchFx];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
fx_t* g_scratch_ptr[kMaxDevices] = {};
// A failed call could not clear the flag either: the next one does so first.
std::atomic<bool> g_flag_left[kMaxDevices];

struct Partials {
    fx_t *inner, *mass, *term;   // kNoAllocBlocks each
    fx_t* bad;
};

// Clears a[0, nv), and sets the flag when a row is not part of the arc
// arrays or a community is out of range.
__global__ void __launch_bounds__(kBlock)
na_check_kernel(const int64_t* __restrict__ off, const int64_t* __restrict__ comm, int64_t nv, int64_t ne,
                fx_t* __restrict__ a, fx_t* __restrict__ flag)
{
    bool bad = false;
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < nv; i += (int64_t)gridDim.x * kBlock) {
        a[i] = 0;
        const int64_t e0 = off[i], e1 = off[i + 1], c = comm[i];
        bad |= e0 < 0 || e1 > ne || e0 > e1 || c < 0 || c >= nv;
    }
    if (bad) *flag = 1;   // every writer stores the same value
}

// k_v (self arcs included, graph_cuda.cu:302-346) into a[comm[v]], the weight
// of arcs whose ends share a community (self arcs included) into P.inner, and
// every weight into P.mass.  Arc-parallel: a workgroup takes tiles of
// kNaTile consecutive arcs and a thread kNaRun consecutive ones of them, whose
// loads and comm gathers are all in flight before the first is used; the rows
// of the tile are found once per workgroup (64-way searches of the first and
// the last, then kNaRows offsets at a time in LDS) and a thread walks them
// forward.  The weights of a thread's part of a row are summed in registers,
// then per community in an LDS table, so a community takes one global atomic
// per tile.  A tile that spans more than kNaSpan rows, most of them empty, has
// every thread search for its own arcs' rows instead.  Exact integer sums:
// neither the split nor the order changes them.  Bound by the comm gathers and
// by the loads of a thread's run, whose lanes lie 64 bytes apart; four waves a
// SIMD (128 registers, 48 bytes of scratch) hide them better than the three
// that 162 registers allow, and better than five (96 registers, 112 bytes: 197
// us).  A call on 2^20 vertices, 14.7 M arcs in planted blocks: 150 us, 180 with
// three waves, 157 without the loads of 16 bytes; 544 us with a wavefront per
// row (a quarter of its lanes busy, a 128-bit wavefront sum and two global
// atomics per row).  An id outside [0, nv)
// is never used as an index: it sets the flag; with the flag set by
// na_check_kernel nothing is read.
constexpr int kNaRun = 8, kNaTile = kBlock * kNaRun, kNaRows = 512, kNaSlots = 2 * kNaRows, kNaSpan = 8 * kNaRows;
__global__ void __launch_bounds__(kBlock, 4)
na_arcs_kernel(const int64_t* __restrict__ off, const int64_t* __restrict__ col, const double* __restrict__ w,
               const int64_t* __restrict__ comm, int64_t nv, fx_t* __restrict__ a, Partials P)
{
    __shared__ int key[kNaSlots];
    __shared__ unsigned long long lo[kNaSlots], hi[kNaSlots];
    __shared__ int s_off[kNaRows + 1], s_comm[kNaRows], s_slot[kNaRows];
    __shared__ fx_t red[kBlock / 64];
    __shared__ int64_t s_row[2];
    // Set by na_check_kernel.  A workgroup that sees it set by another one of
    // this launch (an arc id out of range) may leave as well: Q is NaN then.
    __shared__ int s_bad;
    if (threadIdx.x == 0) s_bad = ld_u64_agent(reinterpret_cast<const unsigned long long*>(P.bad)) != 0;
    __syncthreads();
    if (s_bad) return;
    const int64_t A0 = off[0], A1 = off[nv];
    fx_t I = 0, M = 0;
    bool bad = false;
    for (int64_t t0 = A0 + (int64_t)blockIdx.x * kNaTile; t0 < A1; t0 += (int64_t)gridDim.x * kNaTile) {
        const int n = (int)(t0 + kNaTile < A1 ? kNaTile : A1 - t0);
        for (int s = threadIdx.x; s < kNaSlots; s += kBlock) {
            key[s] = -1;
            lo[s] = 0;
            hi[s] = 0;
        }
        if (threadIdx.x < 128) {                     // wavefront 0: the first row, 1: the last
            const int last = threadIdx.x >> 6;
            const int64_t r = wave_row_of(off, 0, nv, last ? t0 + n - 1 : t0);
            if ((threadIdx.x & 63) == 0) s_row[last] = r;
        }
        const int x0 = threadIdx.x * kNaRun;
        int64_t u[kNaRun];
        double wt[kNaRun];
        int cu[kNaRun];
        if (n == kNaTile) {                          // uniform: loads of 16 bytes
#pragma unroll
            for (int j = 0; j < kNaRun; ++j) u[j] = col[t0 + x0 + j];
#pragma unroll
            for (int j = 0; j < kNaRun; ++j) wt[j] = w[t0 + x0 + j];
        } else {
#pragma unroll
            for (int j = 0; j < kNaRun; ++j) {
                u[j] = x0 + j < n ? col[t0 + x0 + j] : 0;
                wt[j] = x0 + j < n ? w[t0 + x0 + j] : 0.0;
            }
        }
#pragma unroll
        for (int j = 0; j < kNaRun; ++j) {
            const bool ok = u[j] >= 0 && u[j] < nv;
            bad |= !ok;
            cu[j] = ok ? (int)comm[u[j]] : -1;
        }
        __syncthreads();
        const int64_t rf = s_row[0], span = s_row[1] - rf + 1;
        if (span > kNaSpan) {                        // uniform
            if (x0 < n) {
                int row[kNaRun];
                rows_of<kNaRun>(off, rf, (int)span, t0 + x0, t0 + n - 1, row);
                fx_t k = 0;
#pragma unroll
                for (int j = 0; j < kNaRun; ++j) {
                    if (x0 + j >= n) break;
                    const int64_t c = comm[rf + row[j]];
                    asm volatile("" : "+v"(wt[j]));      // keeps the eight conversions apart
                    const fx_t f = fx_from_double(wt[j]);
                    k += f;
                    M += f;
                    if (cu[j] == c) I += f;
                    if (j + 1 < kNaRun && x0 + j + 1 < n && row[j + 1] == row[j]) continue;
                    acc_add(a + c, k);
                    k = 0;
                }
            }
            __syncthreads();                         // the table and s_row are reused
            continue;
        }
        for (int64_t r0 = rf; r0 < rf + span; r0 += kNaRows) {   // uniform: kNaRows rows at a time
            for (int q = threadIdx.x; q <= kNaRows; q += kBlock) {
                const int64_t at = (r0 + q < nv ? off[r0 + q] : A1) - t0;
                s_off[q] = at < 0 ? 0 : at < n ? (int)at : n;
            }
            __syncthreads();
            for (int q = threadIdx.x; q < kNaRows; q += kBlock)
                if (s_off[q] < s_off[q + 1]) {       // a row with arcs in this tile
                    const int c = (int)comm[r0 + q];
                    s_comm[q] = c;
                    s_slot[q] = lds_slot<kNaSlots>(key, c);
                }
            __syncthreads();
            const int c0 = s_off[0], c1 = s_off[kNaRows];
            int l = -1;                              // the row of the arc before
            fx_t k = 0;
#pragma unroll
            for (int j = 0; j < kNaRun; ++j) {
                const int x = x0 + j;
                if (x < c0 || x >= c1) continue;
                if (l < 0) {
                    l = 0;
#pragma unroll
                    for (int st = kNaRows / 2; st > 0; st >>= 1)
                        if (s_off[l + st] <= x) l += st;
                } else if (s_off[l + 1] <= x) {
                    fx_atomic_add(&lo[s_slot[l]], &hi[s_slot[l]], k);
                    k = 0;
                    do ++l;
                    while (s_off[l + 1] <= x);       // x < c1 = s_off[kNaRows]: ends
                }
                asm volatile("" : "+v"(wt[j]));      // keeps the eight conversions apart
                const fx_t f = fx_from_double(wt[j]);
                k += f;
                M += f;
                if (cu[j] == s_comm[l]) I += f;
            }
            if (l >= 0) fx_atomic_add(&lo[s_slot[l]], &hi[s_slot[l]], k);
            __syncthreads();
            for (int s = threadIdx.x; s < kNaSlots; s += kBlock) {
                const int c = key[s];
                if (c < 0) continue;
                const fx_t x = fx_make(lo[s], (int64_t)hi[s]);
                if (x != 0) acc_add(a + c, x);
                key[s] = -1;
                lo[s] = 0;
                hi[s] = 0;
            }
            __syncthreads();                         // s_off and the table are reused
        }
    }
    I = block_sum_fx(I, red);
    M = block_sum_fx(M, red);
    if (threadIdx.x == 0) {
        P.inner[blockIdx.x] = I;
        P.mass[blockIdx.x] = M;
    }
    if (bad) *P.bad = 1;
}

// The sum of x[0, n) (valid in thread 0).
__device__ __forceinline__ fx_t na_sum(const fx_t* __restrict__ x, int n, fx_t* red)
{
    fx_t t = 0;
    for (int i = threadIdx.x; i < n; i += kBlock) t += x[i];
    return block_sum_fx(t, red);
}

// P.term = partials of the sum over communities of fx((RN(a_c) / 2m)^2), with
// 2m = RN of the n partial masses.
__global__ void __launch_bounds__(kBlock)
na_terms_kernel(const fx_t* __restrict__ a, int64_t nv, Partials P, int n)
{
    __shared__ fx_t red[kBlock / 64];
    __shared__ double s_twom;
    const fx_t m = na_sum(P.mass, n, red);
    if (threadIdx.x == 0) s_twom = fx_to_double(m);
    __syncthreads();
    const double twom_d = s_twom;
    fx_t T = 0;
    if (twom_d != 0.0) {
        for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < nv; i += (int64_t)gridDim.x * kBlock) {
            const double x = fx_to_double(a[i]) / twom_d;
            T += fx_from_double(x * x);
        }
    }
    T = block_sum_fx(T, red);
    if (threadIdx.x == 0) P.term[blockIdx.x] = T;
}

// Q = RN(I) / 2m - RN(T); Q = 0 for a graph without weight, NaN when an id
// was out of range.  Leaves the flag clear for the next call (flags written and
// read within a call instead, by workgroup or wavefront, cost every call 1 to 3
// us, 7% of a small one).
__global__ void __launch_bounds__(kBlock)
na_finish_kernel(Partials P, int n, int nt, double* __restrict__ q)
{
    __shared__ fx_t red[kBlock / 64];
    const fx_t I = na_sum(P.inner, n, red), m = na_sum(P.mass, n, red), T = na_sum(P.term, nt, red);
    if (threadIdx.x == 0) {
        const double twom_d = fx_to_double(m);
        double r = twom_d == 0.0 ? 0.0 : fx_to_double(I) / twom_d - fx_to_double(T);
        if (*P.bad != 0) r = __builtin_nan("");
        *P.bad = 0;
        *q = r;
    }
}

__global__ void na_clear_kernel(fx_t* bad) { *bad = 0; }

// Whether the flag's clearing was launched.
bool clear_flag(fx_t* bad, hipStream_t s)
{
    na_clear_kernel<<<1, 1, 0, s>>>(bad);
    return hipGetLastError() == hipSuccess;
}

// The device address of `scratch` on the current device, resolved once per
// device.
int scratch_address(fx_t** out, int* device)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return set_error(NIDO_ERR_HIP, "hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return set_error(NIDO_ERR_INVALID, "device %d beyond %d", dev, kMaxDevices);
    *device = dev;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return set_error(NIDO_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev,
                             hipGetErrorString(e));
        g_scratch_ptr[dev] = static_cast<fx_t*>(p);
    }
    *out = g_scratch_ptr[dev];
    return NIDO_OK;
}

}  // namespace

extern "C" int nido_modularity_noalloc(int64_t nv, int64_t ne, const int64_t* offsets, const int64_t* cols,
                                       const double* weights, const int64_t* comm, double* q, void* stream)
{
    if (nv < 0 || ne < 0) return set_error(NIDO_ERR_INVALID, "negative size (nv %lld, ne %lld)", (long long)nv,
                                           (long long)ne);
    if (nv > kNoAllocMaxVertices)
        return set_error(NIDO_ERR_CAPACITY, "%lld vertices exceed the %lld this entry point's fixed working "
                         "memory holds", (long long)nv, (long long)kNoAllocMaxVertices);
    if (!q || (nv > 0 && (!offsets || !comm)) || (ne > 0 && (!cols || !weights)))
        return set_error(NIDO_ERR_INVALID, "null array");
    fx_t* base = nullptr;
    int dev = 0;
    int rc = scratch_address(&base, &dev);
    if (rc != NIDO_OK) return rc;
    fx_t* a = base;
    fx_t* part = base + kNoAllocMaxVertices;
    const Partials P{part, part + kNoAllocBlocks, part + 2 * kNoAllocBlocks, part + 3 * kNoAllocBlocks};
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (g_flag_left[dev].load() && clear_flag(P.bad, s)) {
        hipStreamCaptureStatus st = hipStreamCaptureStatusActive;   // captured: cleared at the replay only
        if (hipStreamIsCapturing(s, &st) == hipSuccess && st == hipStreamCaptureStatusNone) g_flag_left[dev] = false;
    }
    const unsigned nt = grid_for(nv, kBlock, 1024);
    unsigned n = 0;
    na_check_kernel<<<grid_for(nv, kBlock, 2048), kBlock, 0, s>>>(offsets, comm, nv, ne, a, P.bad);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) {   // what was not checked is not read
        if (nv > 0 && ne > 0) {
            n = grid_for(ne, kNaTile, kNoAllocBlocks);
            na_arcs_kernel<<<n, kBlock, 0, s>>>(offsets, cols, weights, comm, nv, a, P);
        }
        na_terms_kernel<<<nt, kBlock, 0, s>>>(a, nv, P, (int)n);
        na_finish_kernel<<<1, kBlock, 0, s>>>(P, (int)n, (int)nt, q);
        e = hipGetLastError();
        if (e != hipSuccess && !clear_flag(P.bad, s)) g_flag_left[dev] = true;
    }
    if (e != hipSuccess) return set_error(NIDO_ERR_HIP, "nido_modularity_noalloc launch: %s", hipGetErrorString(e));
    return NIDO_OK;
}
