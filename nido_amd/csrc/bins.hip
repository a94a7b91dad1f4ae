// bins.hip -- per-phase work lists built on the device for large phases:
// the degree bins of every batch (rows grouped by (batch, bin), ascending id
// inside a group, isolated vertices left out).  The same lists as the host
// builder (host_bins.cpp), by stable counting sorts over tiles of consecutive
// vertices.
#include "device_common.h"

namespace nido {
namespace {

// The bin of a row of d > 0 arcs (bin_of in host_bins.cpp).
__device__ __forceinline__ int dev_bin(int64_t d, int thread_max, int64_t big_min)
{
    if (d > big_min) return BIN_BIG;
    if (d <= thread_max) return BIN_THREAD;
    if (d <= kBinMaxDeg[BIN_G8]) return BIN_G8;
    if (d <= kBinMaxDeg[BIN_G16]) return BIN_G16;
    if (d <= kBinMaxDeg[BIN_G32]) return BIN_G32;
    if (d <= kBinMaxDeg[BIN_G64]) return BIN_G64;
    if (d <= kBinMaxDeg[BIN_B256]) return BIN_B256;
    return BIN_BIG;
}

// Per tile: its rows of each bin, at cnt[at + k * stride].
__global__ void __launch_bounds__(kBlock)
bin_count_kernel(const BinTile* __restrict__ tiles, int64_t ntiles, const int64_t* __restrict__ off, int thread_max,
                 int64_t big_min, int64_t* __restrict__ cnt)
{
    __shared__ int c[NUM_BINS];
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const BinTile T = tiles[t];
        if (threadIdx.x < NUM_BINS) c[threadIdx.x] = 0;
        __syncthreads();
        for (int64_t v = T.v0 + threadIdx.x; v < T.v1; v += kBlock) {
            const int64_t d = off[v + 1] - off[v];
            if (d > 0) atomicAdd(&c[dev_bin(d, thread_max, big_min)], 1);
        }
        __syncthreads();
        if (threadIdx.x < NUM_BINS) cnt[T.at + threadIdx.x * T.stride] = c[threadIdx.x];
        __syncthreads();   // c is cleared for the next tile
    }
}

// Per tile: every row written at base[at + k * stride] plus its rank among
// the tile's earlier rows of bin k, so each (batch, bin) group lists its rows
// in ascending id.
__global__ void __launch_bounds__(kBlock)
bin_scatter_kernel(const BinTile* __restrict__ tiles, int64_t ntiles, const int64_t* __restrict__ off, int thread_max,
                   int64_t big_min, const int64_t* __restrict__ base, BinRow* __restrict__ binv)
{
    __shared__ int wc[kBlock / 64][NUM_BINS];   // this pass's rows per wavefront and bin
    __shared__ int run[NUM_BINS];               // rows of the tile's earlier passes per bin
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const BinTile T = tiles[t];
        if (threadIdx.x < NUM_BINS) run[threadIdx.x] = 0;
        __syncthreads();
        for (int64_t r0 = T.v0; r0 < T.v1; r0 += kBlock) {   // uniform; one pass per kBlock rows
            const int64_t v = r0 + threadIdx.x;
            int k = -1;
            int64_t d = 0, e0 = 0;
            if (v < T.v1) {
                e0 = off[v];
                d = off[v + 1] - e0;
                if (d > 0) k = dev_bin(d, thread_max, big_min);
            }
            int rank = 0;
#pragma unroll
            for (int kk = 0; kk < NUM_BINS; ++kk) {
                const unsigned long long m = __ballot(k == kk);
                if (k == kk) rank = __popcll(m & below);
                if (lane == 0) wc[wv][kk] = __popcll(m);
            }
            __syncthreads();
            if (k >= 0) {
                int before = run[k];
                for (int i = 0; i < wv; ++i) before += wc[i][k];
                binv[base[T.at + k * T.stride] + before + rank] =
                    BinRow{(int)v, (int)(d < INT32_MAX ? d : INT32_MAX), e0};
            }
            __syncthreads();   // run and wc read before they change
            if (threadIdx.x < NUM_BINS) {
                int s = 0;
                for (int i = 0; i < kBlock / 64; ++i) s += wc[i][threadIdx.x];
                run[threadIdx.x] += s;
            }
            __syncthreads();
        }
    }
}

// out[b * NUM_BINS + k] = the first position of group (b, k), or -1 for a
// batch without tiles.
__global__ void __launch_bounds__(kBlock)
bin_starts_kernel(const int64_t* __restrict__ base, const int64_t* __restrict__ tb0, int nb, int64_t* __restrict__ out)
{
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < nb * NUM_BINS; i += gridDim.x * kBlock) {
        const int b = i / NUM_BINS, k = i % NUM_BINS;
        const int64_t n = tb0[b + 1] - tb0[b];
        out[i] = n > 0 ? base[NUM_BINS * tb0[b] + k * n] : -1;
    }
}

}  // namespace

void launch_bin_count(const BinTile* tiles, int64_t ntiles, const int64_t* off, int thread_max, int64_t big_min,
                      int64_t* cnt, hipStream_t s)
{
    if (ntiles > 0)
        bin_count_kernel<<<grid_for(ntiles, 1, 8192), kBlock, 0, s>>>(tiles, ntiles, off, thread_max, big_min, cnt);
}

void launch_bin_scatter(const BinTile* tiles, int64_t ntiles, const int64_t* off, int thread_max, int64_t big_min,
                        const int64_t* base, BinRow* binv, hipStream_t s)
{
    if (ntiles > 0)
        bin_scatter_kernel<<<grid_for(ntiles, 1, 8192), kBlock, 0, s>>>(tiles, ntiles, off, thread_max, big_min,
                                                                          base, binv);
}

void launch_bin_starts(const int64_t* base, const int64_t* tb0, int nb, int64_t* out, hipStream_t s)
{
    if (nb > 0) bin_starts_kernel<<<grid_for((int64_t)nb * NUM_BINS, kBlock), kBlock, 0, s>>>(base, tb0, nb, out);
}

}  // namespace nido
