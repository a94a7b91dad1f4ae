// kernels.hip -- per-phase and per-iteration kernels other than local moving:
// vertex weights and 2m, singleton partition, modularity, exclusive scan and
// the coarsening (renumber + coarse CSR rebuild) of the batched Louvain path.
#include "device_common.h"

namespace nido {
namespace {

// p[i] = i.
__global__ void iota_kernel(int64_t* __restrict__ p, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) p[i] = i;
}

template <typename T>
__global__ void fill_kernel(T* __restrict__ p, T val, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock)
        p[i] = val;
}

// ---------------------------------------------------------------------------
// Vertex weights (graph_cuda.cu:302-346), singleton (graph_cuda.cu:410-429)
// ---------------------------------------------------------------------------
// Adds a lane's view of the weights to the whole: the largest fractional bits
// and magnitude, and flags.  A wavefront that has nothing new leaves the
// memory alone: atomics on one address take their turn, about 10 ns each, and
// 8,192 wavefronts' made most of this pass (R-MAT scale 20, 60 M arcs: 194 us
// with them, a tenth of that read time).
__device__ __forceinline__ void join_grid(WeightGrid* G, int f, unsigned long long mx, unsigned flags)
{
#pragma unroll
    for (int msk = 32; msk > 0; msk >>= 1) {
        const int of = __shfl_xor(f, msk, 64);
        const unsigned long long om = __shfl_xor(mx, msk, 64);
        f = of > f ? of : f;
        mx = om > mx ? om : mx;
        flags |= __shfl_xor(flags, msk, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        if (f > ld_i32_agent(&G->fneed)) atomicMax(&G->fneed, f);
        if (mx > ld_u64_agent(&G->wmax)) atomicMax(&G->wmax, mx);
        if (flags & ~(unsigned)ld_i32_agent(&G->flags)) atomicOr(&G->flags, (int)flags);
    }
}

// The fractional bits a weight needs (w = sig 2^(ex - 1075), lowest set bit
// 2^(ex - 1075 + ctz(sig)); 2000 for a subnormal or non-finite weight), given
// the bits b of |w|, not zero.
__device__ __forceinline__ int bits_needed(unsigned long long b)
{
    const int ex = (int)(b >> 52);
    if (ex == 0 || ex == 0x7ff) return 2000;
    return 1075 - ex - __builtin_ctzll((b & 0x000fffffffffffffull) | 0x0010000000000000ull);
}

// k (zeroed by the caller) and src[e] = the row of arc e, and the grid of the
// weights, in one pass over the arcs: a workgroup takes tiles of kSumTile
// consecutive arcs and a thread kSumRun consecutive ones of them.  The first
// and the last row of a tile are found by 64-way searches.  Where at most
// kSumSpan rows lie between them, the workgroup takes kSumRows offsets at a
// time into LDS and a thread walks them forward, summing a row's arcs in
// registers and then in LDS; a row inside the tile is stored, a row that
// crosses its ends added with one atomic.  Where more lie between them, most
// have no arcs (coarse graphs of R-MAT: ten without for one with some): every
// thread then searches for the rows of its own arcs and adds a row's sum to k.
// Walking such tiles through LDS as well took one of them to 3.9 ms (first
// coarse graph of R-MAT scale 20, 0.03 ms with the search).  Exact integer
// sums: the split does not change them.  No list of rows is needed (the host
// built two per phase, or the device with two round trips), and the weights
// are read once for everything.  R-MAT scale 22 (128 M arcs): 1.22 ms, 1.3 TB/s of
// its 12 B per arc, where the three kernels without the lists took 0.97.  Bound by
// neither memory nor the VALUs (140 instructions an arc keep them 38% busy); what is
// left is the chain of a tile's steps (search, offsets, walk, sums), with the 16
// wavefronts a CU that 40 KB of LDS leave to hide it.
constexpr int kSumRun = 8, kSumTile = kBlock * kSumRun, kSumRows = 2048, kSumSpan = 2 * kSumRows;
__global__ void __launch_bounds__(kBlock)
row_sums_kernel(const int64_t* __restrict__ off, const double* __restrict__ w, int64_t nv, int64_t ne,
                fx_t* __restrict__ k, int* __restrict__ src, WeightGrid* G)
{
    __shared__ int s_off[kSumRows + 1];
    __shared__ unsigned long long lo[kSumRows], hi[kSumRows];
    __shared__ int64_t s_row[2];
    int f = INT_MIN;
    unsigned long long mx = 0;
    for (int64_t t0 = (int64_t)blockIdx.x * kSumTile; t0 < ne; t0 += (int64_t)gridDim.x * kSumTile) {
        const int n = (int)(t0 + kSumTile < ne ? kSumTile : ne - t0);
        if (threadIdx.x < 128) {                 // wavefront 0: the first row, 1: the last
            const int last = threadIdx.x >> 6;
            const int64_t r = wave_row_of(off, 0, nv, last ? t0 + n - 1 : t0);
            if ((threadIdx.x & 63) == 0) s_row[last] = r;
        }
        const int x0 = threadIdx.x * kSumRun;
        double wt[kSumRun];
#pragma unroll
        for (int j = 0; j < kSumRun; ++j) {
            wt[j] = x0 + j < n ? w[t0 + x0 + j] : 0.0;
            const unsigned long long b = nido_dbits(wt[j]) & 0x7fffffffffffffffull;
            if (b == 0) continue;
            const int need = bits_needed(b);
            f = need > f ? need : f;
            mx = b > mx ? b : mx;
        }
        __syncthreads();
        const int64_t rf = s_row[0], span = s_row[1] - rf + 1;
        if (span > kSumSpan) {                   // uniform
            if (x0 < n) {
                int row[kSumRun];
                rows_of<kSumRun>(off, rf, (int)span, t0 + x0, t0 + n - 1, row);
                fx_t sum = 0;
#pragma unroll
                for (int j = 0; j < kSumRun; ++j) {
                    if (x0 + j >= n) break;
                    src[t0 + x0 + j] = (int)(rf + row[j]);
                    sum += fx_from_double(wt[j]);
                    if (j + 1 < kSumRun && x0 + j + 1 < n && row[j + 1] == row[j]) continue;
                    acc_add(k + rf + row[j], sum);
                    sum = 0;
                }
            }
            __syncthreads();                     // s_row is reused by the next tile
            continue;
        }
        for (int64_t r0 = rf; r0 < rf + span; r0 += kSumRows) {   // uniform: kSumRows rows at a time
            for (int q = threadIdx.x; q <= kSumRows; q += kBlock) {
                const int64_t at = (r0 + q < nv ? off[r0 + q] : ne) - t0;
                s_off[q] = at < 0 ? 0 : at < n ? (int)at : n;
            }
            for (int q = threadIdx.x; q < kSumRows; q += kBlock) {
                lo[q] = 0;
                hi[q] = 0;
            }
            __syncthreads();
            const int c0 = s_off[0], c1 = s_off[kSumRows];
            int l = -1;                          // the row of the arc before
            fx_t sum = 0;
#pragma unroll
            for (int j = 0; j < kSumRun; ++j) {
                const int x = x0 + j;
                if (x < c0 || x >= c1) continue;
                if (l < 0) {
                    l = 0;
#pragma unroll
                    for (int st = kSumRows / 2; st > 0; st >>= 1)
                        if (s_off[l + st] <= x) l += st;
                } else if (s_off[l + 1] <= x) {
                    fx_atomic_add(&lo[l], &hi[l], sum);
                    sum = 0;
                    do ++l;
                    while (s_off[l + 1] <= x);   // x < c1 = s_off[kSumRows]: ends
                }
                sum += fx_from_double(wt[j]);
                src[t0 + x] = (int)(r0 + l);
            }
            if (l >= 0) fx_atomic_add(&lo[l], &hi[l], sum);
            __syncthreads();
            for (int q = threadIdx.x; q < kSumRows; q += kBlock) {
                if (s_off[q] >= s_off[q + 1]) continue;   // no arcs in this tile
                const int64_t r = r0 + q;
                const fx_t x = fx_make(lo[q], (int64_t)hi[q]);
                if (off[r] >= t0 && off[r + 1] <= t0 + n) k[r] = x;
                else acc_add(k + r, x);
            }
            __syncthreads();                     // s_off and the sums are reused
        }
    }
    join_grid(G, f, mx, 0);
}

// kd = FP64(k); part[block] = this block's sum of k; *maxabs = max |kd| as
// raw bits (|x| bit patterns order like the values).
__global__ void __launch_bounds__(kBlock)
round_kernel(const fx_t* __restrict__ k, double* __restrict__ kd, int64_t n,
             unsigned long long* maxabs, fx_t* __restrict__ part)
{
    __shared__ fx_t red[kBlock / 64];
    unsigned long long mx = 0;
    fx_t s = 0;
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock) {
        const fx_t ki = k[i];
        const double x = fx_to_double(ki);
        kd[i] = x;
        s += ki;
        const unsigned long long b = nido_dbits(x) & 0x7fffffffffffffffull;
        mx = b > mx ? b : mx;
    }
#pragma unroll
    for (int msk = 32; msk > 0; msk >>= 1) {
        const unsigned long long o = __shfl_xor(mx, msk, 64);
        mx = o > mx ? o : mx;
    }
    if ((threadIdx.x & 63) == 0 && mx > ld_u64_agent(maxabs)) atomicMax(maxabs, mx);
    s = block_sum_fx(s, red);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// out[i] = FP64(x[i]).
__global__ void __launch_bounds__(kBlock)
fx_round_kernel(const fx_t* __restrict__ x, double* __restrict__ out, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        out[i] = fx_to_double(x[i]);
}

// out[0] = sum of part[0..n) (one workgroup).
__global__ void __launch_bounds__(kBlock)
sum_partials_kernel(const fx_t* __restrict__ part, int n, fx_t* out)
{
    __shared__ fx_t red[kBlock / 64];
    fx_t s = 0;
    for (int i = threadIdx.x; i < n; i += kBlock) s += part[i];
    s = block_sum_fx(s, red);
    if (threadIdx.x == 0) *out = s;
}

__global__ void __launch_bounds__(kBlock)
singleton_kernel(int64_t* __restrict__ C, int64_t* __restrict__ Cn, int* __restrict__ C32,
                 fx_t* __restrict__ a, const fx_t* __restrict__ k, int64_t nv)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < nv;
         i += (int64_t)gridDim.x * kBlock) {
        C[i] = i;
        Cn[i] = i;
        C32[i] = (int)i;
        a[i] = k[i];
    }
}

__global__ void __launch_bounds__(kBlock)
widen_kernel(const int* __restrict__ col32, int64_t* __restrict__ col, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock)
        col[i] = col32[i];
}

__global__ void grid_init_kernel(WeightGrid* G)
{
    *G = WeightGrid{0, INT_MIN, 0};
}

__global__ void phase_init_kernel(PhaseOut* out)
{
    out->twom = 0;
    out->maxk = 0;
    out->grid = WeightGrid{0, INT_MIN, 0};
}

// The caller's arcs once they are on the device: ids narrowed into col32, an
// id outside its graph and a negative weight flagged, and the grid of the
// weights, in one pass.  Pieces are parts of one graph's arcs; without a list
// they are the runs of kPieceArcs arcs of the only graph.  Nothing reads an id
// as an index before the host has seen the flags.
__global__ void __launch_bounds__(kBlock)
take_arcs_kernel(const ArcPiece* __restrict__ pieces, int64_t n, int64_t ne, int64_t nv,
                 const int64_t* __restrict__ col, const double* __restrict__ w, int* __restrict__ col32, WeightGrid* G)
{
    int f = INT_MIN;
    unsigned long long mx = 0;
    unsigned flags = 0;
    for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
        const int64_t e = i * kPieceArcs;
        const ArcPiece p = pieces ? pieces[i] : ArcPiece{e, e + kPieceArcs < ne ? e + kPieceArcs : ne, 0, nv};
        for (int64_t j = p.e0 + threadIdx.x; j < p.e1; j += kBlock) {
            const int64_t c = col[j];
            const unsigned long long x = nido_dbits(w[j]), b = x & 0x7fffffffffffffffull;
            col32[j] = (int)c;
            if (c < p.base || c >= p.base + p.nv) flags |= kArcOutside;
            if (b == 0) continue;
            if (x != b) flags |= kArcNegative;
            const int need = bits_needed(b);
            f = need > f ? need : f;
            mx = b > mx ? b : mx;
        }
    }
    join_grid(G, f, mx, flags);
}

// wq[e] = w[e] * 2^F, exact: every weight is a multiple of 2^-F and
// |w| 2^F < 2^63 (checked by the caller).
__global__ void __launch_bounds__(kBlock)
to_fixed_kernel(const double* __restrict__ w, int64_t* __restrict__ wq, int64_t ne, double scale)
{
    for (int64_t e = blockIdx.x * (int64_t)kBlock + threadIdx.x; e < ne; e += (int64_t)gridDim.x * kBlock)
        wq[e] = (int64_t)(w[e] * scale);
}

// ---------------------------------------------------------------------------
// Modularity (graph_cuda.cu:2078-2134): Q = I/(2m) - sum_c (a_c/(2m))^2.
// Arc-parallel over the whole CSR (tiles of 256 x kModUnroll arcs, every load
// coalesced except the two C gathers), then the community sweep; each block
// leaves two partials and mod_finalize_kernel adds them up.  Ident: C is
// the identity (the singleton partition every phase starts from), so an arc
// is internal exactly when it is a self arc and the C gathers are left out;
// the sums are the same integers either way.
// ---------------------------------------------------------------------------
constexpr int kModUnroll = 8;

template <bool Ident>
__global__ void __launch_bounds__(kBlock)
mod_kernel(const int* __restrict__ src, const int* __restrict__ col,
           const double* __restrict__ w, const int* __restrict__ C, int64_t ne,
           const fx_t* __restrict__ a, int64_t nv, double twom_d, fx_t* __restrict__ part,
           fx_t* __restrict__ term)
{
    __shared__ fx_t red[kBlock / 64];
    fx_t I = 0, T = 0;
    const int64_t tile = (int64_t)kBlock * kModUnroll;
    for (int64_t t0 = blockIdx.x * tile; t0 < ne; t0 += (int64_t)gridDim.x * tile) {
        int s[kModUnroll];
        int u[kModUnroll];
#pragma unroll
        for (int j = 0; j < kModUnroll; ++j) {
            const int64_t e = t0 + j * kBlock + threadIdx.x;
            s[j] = e < ne ? src[e] : 0;
            u[j] = e < ne ? col[e] : 0;
        }
        bool in[kModUnroll];
#pragma unroll
        for (int j = 0; j < kModUnroll; ++j) {
            const int64_t e = t0 + j * kBlock + threadIdx.x;
            if constexpr (Ident) in[j] = e < ne && s[j] == u[j];
            else in[j] = e < ne && C[s[j]] == C[u[j]];    // self arcs are internal
        }
#pragma unroll
        for (int j = 0; j < kModUnroll; ++j)
            if (in[j]) I += fx_from_double(w[t0 + j * kBlock + threadIdx.x]);
    }
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < nv;
         i += (int64_t)gridDim.x * kBlock) {
        const double x = fx_to_double(a[i]) / twom_d;
        const fx_t t = fx_from_double(x * x);
        T += t;
        if (term) term[i] = t;
    }
    I = block_sum_fx(I, red);
    T = block_sum_fx(T, red);
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = I;
        part[2 * blockIdx.x + 1] = T;
    }
}

__global__ void __launch_bounds__(kBlock)
mod_finalize_kernel(const fx_t* __restrict__ part, int nblocks, double twom_d, double* q, fx_t* acc)
{
    __shared__ fx_t red[kBlock / 64];
    fx_t I = 0, T = 0;
    for (int i = threadIdx.x; i < nblocks; i += kBlock) {
        I += part[2 * i];
        T += part[2 * i + 1];
    }
    I = block_sum_fx(I, red);
    T = block_sum_fx(T, red);
    if (threadIdx.x == 0) {
        *q = fx_to_double(I) / twom_d - fx_to_double(T);
        if (acc) {
            acc[0] = I;
            acc[1] = T;
        }
    }
}

// Modularity of a phase whose arcs stream through a window: the internal
// weight of rows [v0, v1) (col / w may be based so that the window's arcs
// keep their CSR indices), added exactly into acc[0]; then every
// community's square term into acc[1]; then Q.  Each thread takes runs of
// kModRun consecutive arcs of [off[v0], off[v1]): a binary search over
// off[v0 .. v1 - 1] finds the row of a run's first arc, then the run walks
// the rows forward, so a long row is spread over many threads and short
// rows leave no lane idle.
constexpr int kModRun = 16;

__global__ void __launch_bounds__(kBlock)
mod_rows_kernel(const int64_t* __restrict__ off, const int* __restrict__ col, const double* __restrict__ w,
                const int* __restrict__ C, int64_t v0, int64_t v1, fx_t* __restrict__ acc)
{
    __shared__ fx_t red[kBlock / 64];
    const int64_t e0 = off[v0], e1 = off[v1];
    fx_t I = 0;
    for (int64_t a = e0 + (blockIdx.x * (int64_t)kBlock + threadIdx.x) * kModRun; a < e1;
         a += (int64_t)gridDim.x * kBlock * kModRun) {
        // the last row r of [v0, v1) with off[r] <= a: off[v0] <= a < off[v1]
        int64_t lo = v0, hi = v1 - 1;
        while (lo < hi) {
            const int64_t mid = lo + (hi - lo + 1) / 2;
            if (off[mid] <= a) lo = mid;
            else hi = mid - 1;
        }
        int64_t r = lo, rend = off[r + 1];
        int cv = C[r];
        const int64_t z = a + kModRun < e1 ? a + kModRun : e1;
        for (int64_t e = a; e < z; ++e) {
            while (rend <= e) {   // e < off[v1]: r stays below v1
                ++r;
                rend = off[r + 1];
                cv = C[r];
            }
            if (C[col[e]] == cv) I += fx_from_double(w[e]);   // self arcs are internal
        }
    }
    I = block_sum_fx(I, red);
    if (threadIdx.x == 0 && I != 0) acc_add(acc, I);
}

__global__ void __launch_bounds__(kBlock)
mod_terms_kernel(const fx_t* __restrict__ a, int64_t nv, double twom_d, fx_t* __restrict__ acc,
                 fx_t* __restrict__ term)
{
    __shared__ fx_t red[kBlock / 64];
    fx_t T = 0;
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < nv; i += (int64_t)gridDim.x * kBlock) {
        const double x = fx_to_double(a[i]) / twom_d;
        const fx_t t = fx_from_double(x * x);
        if (term) term[i] = t;
        T += t;
    }
    T = block_sum_fx(T, red);
    if (threadIdx.x == 0 && T != 0) acc_add(acc + 1, T);
}

__global__ void mod_acc_finish_kernel(const fx_t* __restrict__ acc, double twom_d, double* q)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *q = fx_to_double(acc[0]) / twom_d - fx_to_double(acc[1]);
}

// The multisets {(src, dst, w)} and {(dst, src, w)} of the arcs, compared
// through sums (mod 2^64) of two keyed hashes of each form: equal when every
// arc has a reverse arc of the same weight, and unequal otherwise except
// with probability about 2^-128.  The mixer is the output function of
// splitmix64 (Vigna's public-domain splitmix64.c; Stafford's "Mix13"
// constants); the two keys are the first 64 fraction bits of sqrt(2) and
// sqrt(3).
__device__ __forceinline__ unsigned long long mix64(unsigned long long z)
{
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

__device__ __forceinline__ unsigned long long arc_hash(unsigned a, unsigned b, unsigned long long wb,
                                                       unsigned long long key)
{
    return mix64(mix64((((unsigned long long)a << 32) | b) ^ key) ^ wb);
}

// Each workgroup leaves its four sums in part; sym_sum_kernel adds them up
// (8,192 wavefronts adding to the same four words took 320 us whatever the
// size of the graph, 546 us for 60 M arcs).
__global__ void __launch_bounds__(kBlock)
sym_hash_kernel(const int* __restrict__ src, const int* __restrict__ col, const double* __restrict__ w, int64_t ne,
                unsigned long long* __restrict__ part)
{
    constexpr unsigned long long k1 = 0x6a09e667f3bcc909ull, k2 = 0xbb67ae8584caa73bull;
    __shared__ unsigned long long red[4][kBlock / 64];
    unsigned long long h[4] = {0, 0, 0, 0};
    for (int64_t e = blockIdx.x * (int64_t)kBlock + threadIdx.x; e < ne; e += (int64_t)gridDim.x * kBlock) {
        const unsigned a = (unsigned)src[e], b = (unsigned)col[e];
        const unsigned long long wb = (unsigned long long)__double_as_longlong(w[e]);
        h[0] += arc_hash(a, b, wb, k1);
        h[1] += arc_hash(b, a, wb, k1);
        h[2] += arc_hash(a, b, wb, k2);
        h[3] += arc_hash(b, a, wb, k2);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int msk = 32; msk > 0; msk >>= 1) h[i] += __shfl_xor(h[i], msk, 64);
        if ((threadIdx.x & 63) == 0) red[i][threadIdx.x >> 6] = h[i];
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        unsigned long long t = 0;
        for (int i = 0; i < kBlock / 64; ++i) t += red[threadIdx.x][i];
        part[4 * (int64_t)blockIdx.x + threadIdx.x] = t;
    }
}

// out[i] = the sum of part[4 j + i] over the n workgroups j (a wavefront per i).
__global__ void __launch_bounds__(kBlock)
sym_sum_kernel(const unsigned long long* __restrict__ part, int n, unsigned long long* __restrict__ out)
{
    static_assert(kBlock / 64 == 4, "a wavefront per sum");
    const int i = threadIdx.x >> 6;
    unsigned long long t = 0;
    for (int j = threadIdx.x & 63; j < n; j += 64) t += part[4 * j + i];
#pragma unroll
    for (int msk = 32; msk > 0; msk >>= 1) t += __shfl_xor(t, msk, 64);
    if ((threadIdx.x & 63) == 0) out[i] = t;
}

__global__ void __launch_bounds__(kBlock)
mod_delta_kernel(int b, int64_t v0, int64_t v1, const int64_t* __restrict__ Cn, const int* __restrict__ C32,
                 const int* __restrict__ col, const double* __restrict__ w, const fx_t* __restrict__ a,
                 double twom_d, ModDelta D)
{
    __shared__ fx_t red[kBlock / 64];
    delta_body(b, v0, v1, Cn, C32, col, w, a, twom_d, D, (int)blockIdx.x, (int)gridDim.x, red);
}

__global__ void __launch_bounds__(kBlock)
mod_finish_kernel(ModDelta D, int nb, double twom_d, double* q)
{
    if (threadIdx.x == 0 && blockIdx.x == 0)
        *q = fx_to_double(D.acc[0]) / twom_d - fx_to_double(D.acc[1]);
    for (int i = threadIdx.x; i < 2 * nb; i += kBlock) D.counts[i] = 0;
}

// Per graph: the graphs that sat out keep their last q[g] (and their
// accumulators describe no partition once they have been rolled back).
__global__ void __launch_bounds__(kBlock)
mod_finish_graphs_kernel(ModDelta D, int nb, int G, double* __restrict__ q, const unsigned char* __restrict__ act)
{
    __shared__ unsigned long long red[kBlock / 64];
    for (int g = blockIdx.x * kBlock + threadIdx.x; g < G; g += gridDim.x * kBlock) {
        if (!act[g]) continue;
        const double tw = D.twomg[g];
        q[g] = tw == 0 ? 0.0 : fx_to_double(D.acc[2 * g]) / tw - fx_to_double(D.acc[2 * g + 1]);
    }
    if (blockIdx.x == 0) {
        for (int i = threadIdx.x; i < 2 * nb; i += kBlock) D.counts[i] = 0;
        if (D.moved) {
            const unsigned long long t = sum_moved_slots(D.moved, red);
            if (threadIdx.x == 0) reinterpret_cast<unsigned long long*>(q)[G] = t;
        }
    }
}

// ---------------------------------------------------------------------------
// Exclusive scan (int64), tiles of 2048 values per 256-thread workgroup;
// blockIdx.y picks one of several arrays, stride apart.
// ---------------------------------------------------------------------------
constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;

__device__ __forceinline__ int64_t block_excl_scan(int64_t x, int64_t* warp_tot, int64_t* total)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int64_t inc = x;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t y = __shfl_up(inc, d, 64);
        if (lane >= d) inc += y;
    }
    if (lane == 63) warp_tot[wv] = inc;
    __syncthreads();
    int64_t pre = 0, all = 0;
#pragma unroll
    for (int i = 0; i < kBlock / 64; ++i) {
        if (i < wv) pre += warp_tot[i];
        all += warp_tot[i];
    }
    *total = all;
    return pre + inc - x;
}

__global__ void __launch_bounds__(kBlock)
scan_tile_sums_kernel(const int64_t* __restrict__ in, int64_t n, int64_t* __restrict__ sums, int64_t stride)
{
    __shared__ int64_t wt[kBlock / 64];
    in += blockIdx.y * stride;
    sums += (int64_t)blockIdx.y * gridDim.x;
    const int64_t t0 = (int64_t)blockIdx.x * kScanTile;
    int64_t s = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        const int64_t i = t0 + (int64_t)j * kBlock + threadIdx.x;
        if (i < n) s += in[i];
    }
    int64_t tot;
    block_excl_scan(s, wt, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(kBlock)
scan_tile_apply_kernel(const int64_t* in, int64_t* out, int64_t n,
                       const int64_t* __restrict__ tile_off, int64_t* total, int64_t stride,
                       int64_t* __restrict__ totals)
{
    __shared__ int64_t wt[kBlock / 64];
    in += blockIdx.y * stride;
    out += blockIdx.y * stride;
    if (tile_off) tile_off += (int64_t)blockIdx.y * gridDim.x;
    if (total) total += blockIdx.y * stride;
    const int64_t t0 = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    int64_t v[kScanItems];
    int64_t s = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        const int64_t i = t0 + j;
        v[j] = i < n ? in[i] : 0;
        s += v[j];
    }
    int64_t tot;
    int64_t run = block_excl_scan(s, wt, &tot) + (tile_off ? tile_off[blockIdx.x] : 0);
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        const int64_t i = t0 + j;
        if (i < n) out[i] = run;
        run += v[j];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == kBlock - 1) {
        if (total) *total = run;
        if (totals) totals[blockIdx.y] = run;
    }
}

// ---------------------------------------------------------------------------
// Coarsening (graph_gpu.cpp:1151-1304, 1382-1545), all on the device.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kBlock)
mark_kernel(const int64_t* __restrict__ C, int64_t nv, int64_t* __restrict__ flag,
            const int* __restrict__ gid, const unsigned char* __restrict__ keep)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < nv;
         i += (int64_t)gridDim.x * kBlock)
        if (!gid || keep[gid[i]]) flag[C[i]] = 1;
}

__global__ void __launch_bounds__(kBlock)
clustering_kernel(int64_t* __restrict__ clus, int64_t n0, const int64_t* __restrict__ C,
                  const int64_t* __restrict__ newid, const int* __restrict__ gid0,
                  const unsigned char* __restrict__ keep)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n0;
         i += (int64_t)gridDim.x * kBlock)
        if (!gid0 || keep[gid0[i]]) clus[i] = newid[C[clus[i]]];
}

__global__ void __launch_bounds__(kBlock)
widen_local_kernel(const ArcPiece* __restrict__ pieces, int64_t n, const uint16_t* __restrict__ local,
                   int* __restrict__ col32)
{
    for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
        const ArcPiece p = pieces[i];
        for (int64_t e = p.e0 + threadIdx.x; e < p.e1; e += kBlock) col32[e] = (int)(p.base + local[e]);
    }
}

// out[i] = clus[i] - base[graph of i]: every graph's clustering in its own
// ids.
__global__ void __launch_bounds__(kBlock)
local_ids_kernel(const int64_t* __restrict__ clus, int64_t n0, const int* __restrict__ gid0,
                 const int64_t* __restrict__ base, int64_t* __restrict__ out)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n0; i += (int64_t)gridDim.x * kBlock)
        out[i] = clus[i] - base[gid0[i]];
}

// The coarse rows of a workgroup's kBlock consecutive vertices are grouped in
// an LDS table: vertices of one community are often neighbours in id, and
// each distinct row then takes one global atomic instead of one per vertex.
constexpr int kGroupSlots = 2 * kBlock;

// cid[v] = the coarse row of vertex v (-1: its graph does not take part),
// and per coarse row its members and arcs.
__global__ void __launch_bounds__(kBlock)
member_counts_kernel(const int64_t* __restrict__ C, const int64_t* __restrict__ newid,
                     const int64_t* __restrict__ off, int64_t nv, int* __restrict__ cid, int64_t* __restrict__ cnt,
                     int64_t* __restrict__ arcs, const int* __restrict__ gid,
                     const unsigned char* __restrict__ keep)
{
    __shared__ int key[kGroupSlots];
    __shared__ unsigned long long nm[kGroupSlots], na[kGroupSlots];
    for (int64_t base = blockIdx.x * (int64_t)kBlock; base < nv; base += (int64_t)gridDim.x * kBlock) {
        for (int s = threadIdx.x; s < kGroupSlots; s += kBlock) {
            key[s] = -1;
            nm[s] = 0;
            na[s] = 0;
        }
        __syncthreads();
        const int64_t v = base + threadIdx.x;
        if (v < nv) {
            const int i = !gid || keep[gid[v]] ? (int)newid[C[v]] : -1;
            cid[v] = i;
            if (i >= 0) {
                const int h = lds_slot<kGroupSlots>(key, i);
                atomicAdd(&nm[h], 1ull);
                atomicAdd(&na[h], (unsigned long long)(off[v + 1] - off[v]));
            }
        }
        __syncthreads();
        for (int s = threadIdx.x; s < kGroupSlots; s += kBlock) {
            const int i = key[s];
            if (i < 0) continue;
            atomicAdd(reinterpret_cast<unsigned long long*>(cnt + i), nm[s]);
            if (na[s]) atomicAdd(reinterpret_cast<unsigned long long*>(arcs + i), na[s]);
        }
        __syncthreads();   // the table is cleared for the next chunk
    }
}

// Whether one wavefront aggregates a coarse row of a arcs and m members: each
// lane takes one member, then one arc.  Members without arcs count: a vertex
// that only has arcs towards it, as one-way inputs give, joins no community but
// others join its own, so a row has up to a + 1 members.
__device__ __forceinline__ bool wave_row(int64_t a, int64_t m)
{
    return a <= kWaveRowArcs && m <= kWaveRowArcs;
}

// Coarse row i with arcs[i] <= kLdsRowArcs is aggregated in LDS and needs
// csz[i] = min(arcs, K) compact entries; a longer one gets an HBM hash table
// of tsz[i] slots (a power of two >= twice its possible keys, whole words of
// kSlotWord slots).  ml / mh: the members of LDS and of HBM rows.  The LDS
// rows of more arcs or members than a wavefront has lanes are listed in mid[0,
// *nmid).
__global__ void __launch_bounds__(kBlock)
coarse_sizes_kernel(const int64_t* __restrict__ arcs, const int64_t* __restrict__ cnt, int64_t K,
                    int64_t* __restrict__ ml, int64_t* __restrict__ mh, int64_t* __restrict__ tsz,
                    int64_t* __restrict__ csz, int* __restrict__ mid, unsigned long long* __restrict__ nmid)
{
    for (int64_t b = blockIdx.x * (int64_t)kBlock; b < K; b += (int64_t)gridDim.x * kBlock) {
        const int64_t i = b + threadIdx.x;
        bool listed = false;
        if (i < K) {
            const int64_t a = arcs[i], m = cnt[i];
            const int64_t need = a < K ? a : K;
            const bool hbm = a > kLdsRowArcs;
            int64_t s = 0;
            if (hbm) {
                s = kSlotWord;
                while (s < 2 * need) s <<= 1;
            }
            tsz[i] = s;
            csz[i] = hbm ? 0 : need;
            ml[i] = hbm ? 0 : m;
            mh[i] = hbm ? m : 0;
            listed = !hbm && !wave_row(a, m);
        }
        const unsigned long long w = __ballot(listed);
        if (w) {   // uniform in the wavefront
            unsigned long long at = 0;
            if ((threadIdx.x & 63) == 0) at = atomicAdd(nmid, (unsigned long long)__popcll(w));
            at = __shfl(at, 0, 64);
            if (listed) mid[at + __popcll(w & ((1ull << (threadIdx.x & 63)) - 1))] = (int)i;
        }
    }
}

// members[ml[i] ...) = the vertices of LDS row i and members[ML + mh[i] ...)
// those of HBM row i (ML = ml[K]), in no set order inside a row; hd gets the
// degree of every HBM row's member.  Each workgroup reserves a block of its
// rows' member slots with one atomic per distinct row (grouped in LDS as in
// member_counts_kernel).
__global__ void __launch_bounds__(kBlock)
member_scatter_kernel(const int* __restrict__ cid, const int64_t* __restrict__ off, int64_t nv,
                      const int64_t* __restrict__ ml, const int64_t* __restrict__ mh, int64_t ML,
                      const int64_t* __restrict__ toff, unsigned long long* __restrict__ mfill,
                      int* __restrict__ members, int64_t* __restrict__ hd)
{
    __shared__ int key[kGroupSlots];
    __shared__ unsigned nm[kGroupSlots];
    __shared__ unsigned long long at[kGroupSlots];
    for (int64_t base = blockIdx.x * (int64_t)kBlock; base < nv; base += (int64_t)gridDim.x * kBlock) {
        for (int s = threadIdx.x; s < kGroupSlots; s += kBlock) {
            key[s] = -1;
            nm[s] = 0;
        }
        __syncthreads();
        const int64_t v = base + threadIdx.x;
        const int i = v < nv ? cid[v] : -1;
        int h = 0;
        unsigned rank = 0;
        if (i >= 0) {
            h = lds_slot<kGroupSlots>(key, i);
            rank = atomicAdd(&nm[h], 1u);
        }
        __syncthreads();
        for (int s = threadIdx.x; s < kGroupSlots; s += kBlock)
            if (key[s] >= 0) at[s] = atomicAdd(mfill + key[s], (unsigned long long)nm[s]);
        __syncthreads();
        if (i >= 0) {
            const int64_t r = (int64_t)(at[h] + rank);
            if (toff[i + 1] > toff[i]) {
                members[ML + mh[i] + r] = (int)v;
                hd[mh[i] + r] = off[v + 1] - off[v];
            } else {
                members[ml[i] + r] = (int)v;
            }
        }
        __syncthreads();   // the table is cleared for the next chunk
    }
}

// Coarse rows of at most kWaveRowArcs arcs and as many members (wave_row), one
// wavefront each: each lane holds one member, the lengths are scanned with
// shuffles, and each lane then takes one arc and inserts its coarse target into
// the wavefront's 128-slot LDS table.  No workgroup barrier: most coarse rows of a sparse
// graph are this short; bound by the round trips of a row (members, offsets,
// arcs, ids), of which 8,192 wavefronts keep as many in flight.  R-MAT scale
// 20's first coarse graph (316 K rows): 33 us, against 880 us with a
// workgroup per row.
constexpr int kWaveSlots = 2 * (int)kWaveRowArcs;
__global__ void __launch_bounds__(kBlock)
coarse_wave_kernel(const int64_t* __restrict__ arcs, const int64_t* __restrict__ ml,
                   const int* __restrict__ members, const int64_t* __restrict__ off, const int* __restrict__ col,
                   const double* __restrict__ w, const int* __restrict__ cid, int64_t K,
                   const int64_t* __restrict__ cpos, int* __restrict__ ckey, double* __restrict__ cw,
                   int64_t* __restrict__ cnt)
{
    __shared__ int s_key[kBlock / 64][kWaveSlots];
    __shared__ unsigned long long s_lo[kBlock / 64][kWaveSlots], s_hi[kBlock / 64][kWaveSlots];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int* const key = s_key[wv];
    unsigned long long *const lo = s_lo[wv], *const hi = s_hi[wv];
    const int64_t nw = (int64_t)gridDim.x * (kBlock / 64);
    for (int64_t i = (int64_t)blockIdx.x * (kBlock / 64) + wv; i < K; i += nw) {   // uniform in the wavefront
        const int64_t a = arcs[i], m0 = ml[i], m = ml[i + 1] - m0;
        if (!wave_row(a, m)) continue;       // a listed LDS row or an HBM row
        if (a == 0) {
            if (lane == 0) cnt[i] = 0;
            continue;
        }
#pragma unroll
        for (int s = lane; s < kWaveSlots; s += 64) {
            key[s] = -1;
            lo[s] = 0;
            hi[s] = 0;
        }
        const int nm = (int)m;               // <= 64
        int d = 0;
        int64_t e0 = 0;
        if (lane < nm) {
            const int v = members[m0 + lane];
            e0 = off[v];
            d = (int)(off[v + 1] - e0);
        }
        int inc = d;
#pragma unroll
        for (int k = 1; k < 64; k <<= 1) {
            const int y = __shfl_up(inc, k, 64);
            if (lane >= k) inc += y;
        }
        int l = 0;   // the member of this lane's arc: members that end at or before it
#pragma unroll
        for (int sft = 32; sft > 0; sft >>= 1)
            if (__shfl(inc, l + sft - 1, 64) <= lane) l += sft;
        const int start = __shfl(inc, l, 64) - __shfl(d, l, 64);
        const int64_t e = __shfl(e0, l, 64) + (lane - start);
        wave_lds_sync();
        if (lane < a) {
            const int j = cid[col[e]];
            const fx_t x = fx_from_double(w[e]);
            unsigned h = ((unsigned)j * kHashMul) >> (32 - ilog2c(kWaveSlots));
            for (;;) {   // ends: at most 64 of the 128 slots are taken
                const int kk = key[h];
                if (kk == j) break;
                if (kk < 0) {
                    const int prev = atomicCAS(&key[h], -1, j);
                    if (prev < 0 || prev == j) break;
                }
                h = (h + 1) & (kWaveSlots - 1);
            }
            fx_atomic_add(&lo[h], &hi[h], x);
        }
        wave_lds_sync();
        const int64_t base = cpos[i];
        int n = 0;
#pragma unroll
        for (int s0 = 0; s0 < kWaveSlots; s0 += 64) {
            const int s = s0 + lane;
            const int j = key[s];
            const unsigned long long m = __ballot(j >= 0);
            if (j >= 0) {
                const int r = n + __popcll(m & ((1ull << lane) - 1));
                ckey[base + r] = j;
                cw[base + r] = fx_to_double(fx_make(lo[s], (int64_t)hi[s]));
            }
            n += __popcll(m);
        }
        if (lane == 0) cnt[i] = n;
        wave_lds_sync();                     // read before the next row clears the table
    }
}

// The listed coarse rows (at most kLdsRowArcs arcs, more arcs or members than a
// wavefront takes), one workgroup each: the arcs of its members (their concatenation, 256 at a
// time, each thread locating its member by binary search over the scanned
// lengths) go into an LDS table keyed by the coarse target, with exact Q64.64
// sums; the arcs into the row itself are summed per wavefront first and
// inserted once.  The row's distinct targets land compactly at ckey/cw[cpos[i]
// ...) and their count in cnt[i].  Keys whose weights sum to zero are kept,
// as in the HBM tables.
constexpr int kLdsSlots = 2 * kLdsRowArcs;
__global__ void __launch_bounds__(kBlock)
coarse_lds_kernel(const int64_t* __restrict__ arcs, const int64_t* __restrict__ ml,
                  const int* __restrict__ members, const int64_t* __restrict__ off,
                  const int* __restrict__ col, const double* __restrict__ w, const int* __restrict__ cid, int64_t K,
                  const int* __restrict__ mid, const unsigned long long* __restrict__ nmid,
                  const int64_t* __restrict__ cpos, int* __restrict__ ckey, double* __restrict__ cw,
                  int64_t* __restrict__ cnt)
{
    __shared__ int key[kLdsSlots];
    __shared__ unsigned long long lo[kLdsSlots], hi[kLdsSlots];
    __shared__ int klist[kLdsRowArcs];
    __shared__ int s_pre[kBlock], wtot[kBlock / 64];
    __shared__ int64_t s_e0[kBlock];
    __shared__ int s_nk;
    const int lane = threadIdx.x & 63;
    const int64_t n = (int64_t)*nmid;
    for (int64_t t = blockIdx.x; t < n; t += gridDim.x) {
        const int64_t i = mid[t];
        const int64_t a = arcs[i];
        const int64_t need = a < K ? a : K;
        int lg = 6;
        while ((1ll << lg) < 2 * need) ++lg;
        const int ts = 1 << lg;          // <= kLdsSlots
        for (int s = threadIdx.x; s < ts; s += kBlock) {
            key[s] = -1;
            lo[s] = 0;
            hi[s] = 0;
        }
        if (threadIdx.x == 0) s_nk = 0;
        __syncthreads();
        // ends: at most need <= ts / 2 distinct keys
        auto insert = [&](int j, fx_t x) {
            unsigned h = ((unsigned)j * kHashMul) >> (32 - lg);
            for (;;) {
                const int kk = key[h];
                if (kk == j) break;
                if (kk < 0) {
                    const int prev = atomicCAS(&key[h], -1, j);
                    if (prev < 0) {
                        klist[atomicAdd(&s_nk, 1)] = (int)h;
                        break;
                    }
                    if (prev == j) break;
                }
                h = (h + 1) & (unsigned)(ts - 1);
            }
            fx_atomic_add(&lo[h], &hi[h], x);
        };
        fx_t self = 0;
        bool any_self = false;           // uniform in the wavefront
        const int64_t m1 = ml[i + 1];
        for (int64_t m0 = ml[i]; m0 < m1; m0 += kBlock) {   // uniform
            const int64_t mi = m0 + threadIdx.x;
            int d = 0;
            int64_t e0 = 0;
            if (mi < m1) {
                const int v = members[mi];
                e0 = off[v];
                d = (int)(off[v + 1] - e0);   // <= a <= kLdsRowArcs
            }
            int tot;
            const int pre = block_excl_scan_i32(d, wtot, &tot);
            s_pre[threadIdx.x] = pre;
            s_e0[threadIdx.x] = e0;
            __syncthreads();
            const int nm = m1 - m0 < kBlock ? (int)(m1 - m0) : kBlock;
            int top = 1;
            while (2 * top < nm) top *= 2;
            for (int p0 = 0; p0 < tot; p0 += kBlock) {   // uniform
                const int p = p0 + threadIdx.x;
                int j = -1;
                fx_t x = 0;
                if (p < tot) {
                    int l = 0;                 // the last member whose arcs start at or before p
                    for (int st = top; st > 0; st >>= 1)
                        if (l + st < nm && s_pre[l + st] <= p) l += st;
                    const int64_t e = s_e0[l] + (p - s_pre[l]);
                    j = cid[col[e]];
                    x = fx_from_double(w[e]);
                }
                const bool own = j == (int)i;
                any_self |= __ballot(own) != 0;
                if (own) self += x;
                else if (j >= 0) insert(j, x);
            }
            __syncthreads();               // s_pre / s_e0 / wtot are rewritten by the next chunk
        }
        self = wave_sum_fx(self);
        if (lane == 0 && any_self) insert((int)i, self);
        __syncthreads();
        const int nk = s_nk;
        const int64_t base = cpos[i];
        for (int r = threadIdx.x; r < nk; r += kBlock) {
            const int sl = klist[r];
            ckey[base + r] = key[sl];
            cw[base + r] = fx_to_double(fx_make(lo[sl], (int64_t)hi[sl]));
        }
        if (threadIdx.x == 0) cnt[i] = nk;
        __syncthreads();                   // the table is cleared for the next row
    }
}

__device__ __forceinline__ void coarse_insert_one(int64_t i, int j, fx_t wf,
                                                  const int64_t* __restrict__ toff,
                                                  int* __restrict__ tkey, fx_t* __restrict__ tval)
{
    const int64_t base = toff[i];
    const int64_t size = toff[i + 1] - base;
    const int sh = 32 - (63 - __builtin_clzll((unsigned long long)size));
    int* key = tkey + base;
    unsigned long long* val = reinterpret_cast<unsigned long long*>(tval + base);
    uint64_t h = sh >= 32 ? 0 : (((unsigned)j * kHashMul) >> sh);
    for (;;) {
        const int kk = ld_i32_agent(&key[h]);
        if (kk == j) break;
        if (kk < 0) {
            const int prev = atomicCAS(&key[h], -1, j);
            if (prev < 0 || prev == j) break;
        }
        h = (h + 1) & (uint64_t)(size - 1);
    }
    fx_atomic_add(&val[2 * h], &val[2 * h + 1], wf);
}

// The rows with an HBM table: every fine arc (u->x, w) goes into coarse row
// cid[u] under key cid[x]; internal arcs and old self-loops become the coarse
// self-loop (graph_gpu.cpp:1233-1250).  The arcs of these rows' members, in
// member order, are one flat range cut into tiles of kInsTile arcs, one
// workgroup each, so a hub vertex or a giant community costs what its arcs
// cost (R-MAT scale 20's first coarse graph, 60 M arcs: 0.65 ms, against 13.0
// ms with a wavefront per vertex, set by its hubs; a Chung-Lu graph of 8.9 M
// arcs 0.44 against 1.0 ms).  What bounds it now are the LDS atomics of the
// sums and the gathers of cid.  A tile first sums its arcs per (row,
// target) in an LDS table and then adds each sum to the row's HBM table with
// one atomic; an arc that finds no slot within kInsProbe goes to the HBM
// table directly.  The arcs that land in their own row (most of them once
// communities have formed) are summed in registers first.  The sums are
// exact integers, so the grouping does not change them.
constexpr int kInsTile = 4096, kInsSlots = 1024, kInsProbe = 8, kInsUnroll = 4;
__global__ void __launch_bounds__(kBlock)
coarse_insert_kernel(const int64_t* __restrict__ hpre, int64_t n, const int* __restrict__ members,
                     const int* __restrict__ cid, const int64_t* __restrict__ off, const int* __restrict__ col,
                     const double* __restrict__ w, const int64_t* __restrict__ toff, int* __restrict__ tkey,
                     fx_t* __restrict__ tval)
{
    constexpr unsigned long long kEmpty = ~0ull;
    __shared__ unsigned long long key[kInsSlots], lo[kInsSlots], hi[kInsSlots];
    __shared__ int s_pre[kBlock], s_row[kBlock];
    __shared__ int64_t s_e0[kBlock];
    __shared__ int64_t s_m0;
    __shared__ int s_end;
    const int64_t A = hpre[n];
    for (int64_t t0 = (int64_t)blockIdx.x * kInsTile; t0 < A; t0 += (int64_t)gridDim.x * kInsTile) {
        const int64_t t1 = t0 + kInsTile < A ? t0 + kInsTile : A;
        for (int s = threadIdx.x; s < kInsSlots; s += kBlock) {
            key[s] = kEmpty;
            lo[s] = 0;
            hi[s] = 0;
        }
        if (threadIdx.x < 64) {   // the last member whose arcs start at or before t0
            const int64_t l = wave_row_of(hpre, 0, n, t0);
            if (threadIdx.x == 0) s_m0 = l;
        }
        __syncthreads();
        auto insert = [&](int i, int j, fx_t x) {
            const unsigned long long k = ((unsigned long long)(unsigned)i << 32) | (unsigned)j;
            unsigned h = (((unsigned)j ^ ((unsigned)i * kPartMul)) * kHashMul) >> (32 - ilog2c(kInsSlots));
            for (int probe = 0; probe < kInsProbe; ++probe) {
                unsigned long long kk = key[h];
                if (kk == kEmpty) kk = atomicCAS(&key[h], kEmpty, k);
                if (kk == kEmpty || kk == k) {
                    fx_atomic_add(&lo[h], &hi[h], x);
                    return;
                }
                h = (h + 1) & (kInsSlots - 1);
            }
            coarse_insert_one(i, j, x, toff, tkey, tval);
        };
        int own = -1;                      // the row whose self arcs `self` holds
        fx_t self = 0;
        for (int64_t m0 = s_m0;; m0 += kBlock) {   // uniform: chunks of kBlock members
            const int64_t q = m0 + threadIdx.x;
            const int64_t a = q < n ? hpre[q] : A, z = q < n ? hpre[q + 1] : A;
            const int64_t a1 = a < t0 ? t0 : a < t1 ? a : t1;
            s_pre[threadIdx.x] = (int)(a1 - t0);
            if (z > t0 && a < t1 && z > a) {
                const int v = members[q];
                s_e0[threadIdx.x] = off[v] - a;
                s_row[threadIdx.x] = cid[v];
            }
            if (threadIdx.x == kBlock - 1) s_end = (int)((z < t1 ? z : t1) - t0);
            __syncthreads();
            const int c0 = s_pre[0], c1 = s_end;
            for (int x0 = c0; x0 < c1; x0 += kInsUnroll * kBlock) {
                int row[kInsUnroll], tgt[kInsUnroll];
                double wt[kInsUnroll];
#pragma unroll
                for (int r = 0; r < kInsUnroll; ++r) {
                    const int x = x0 + r * kBlock + threadIdx.x;
                    row[r] = -1;
                    tgt[r] = 0;
                    wt[r] = 0.0;
                    if (x < c1) {
                        int l = 0;         // the last member of the chunk whose arcs start at or before x
#pragma unroll
                        for (int st = kBlock / 2; st > 0; st >>= 1)
                            if (s_pre[l + st] <= x) l += st;
                        const int64_t e = s_e0[l] + t0 + x;
                        row[r] = s_row[l];
                        tgt[r] = col[e];
                        wt[r] = w[e];
                    }
                }
#pragma unroll
                for (int r = 0; r < kInsUnroll; ++r)
                    if (row[r] >= 0) tgt[r] = cid[tgt[r]];
#pragma unroll
                for (int r = 0; r < kInsUnroll; ++r) {
                    if (row[r] < 0) continue;
                    const fx_t x = fx_from_double(wt[r]);
                    if (tgt[r] != row[r]) {
                        insert(row[r], tgt[r], x);
                    } else if (own == row[r]) {
                        self += x;
                    } else {
                        if (own >= 0) insert(own, own, self);
                        own = row[r];
                        self = x;
                    }
                }
            }
            __syncthreads();               // the chunk's arrays are rewritten
            if (c1 >= (int)(t1 - t0)) break;   // uniform
        }
        if (own >= 0) insert(own, own, self);
        __syncthreads();
        for (int s = threadIdx.x; s < kInsSlots; s += kBlock) {
            const unsigned long long k = key[s];
            if (k != kEmpty)
                coarse_insert_one((int64_t)(k >> 32), (int)(unsigned)k, fx_make(lo[s], (int64_t)hi[s]), toff, tkey,
                                  tval);
        }
        __syncthreads();                   // the table is cleared for the next tile
    }
}

// HBM tables are whole words of kSlotWord = 64 slots: wcnt[x] = the taken
// slots of word x, one lane per slot.
__global__ void __launch_bounds__(kBlock)
slot_words_kernel(const int* __restrict__ tkey, int64_t nwords, int64_t* __restrict__ wcnt)
{
    const int lane = threadIdx.x & 63;
    const int64_t nw = (int64_t)gridDim.x * (kBlock / 64);
    for (int64_t x = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); x < nwords; x += nw) {
        const unsigned long long m = __ballot(tkey[x * kSlotWord + lane] >= 0);
        if (lane == 0) wcnt[x] = __popcll(m);
    }
}

// cnt[i] = the entries of HBM row i, from the scanned word counts.
__global__ void __launch_bounds__(kBlock)
coarse_count_kernel(const int64_t* __restrict__ toff, const int64_t* __restrict__ wpre, int64_t K,
                    int64_t* __restrict__ cnt)
{
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < K; i += (int64_t)gridDim.x * kBlock) {
        const int64_t a = toff[i], z = toff[i + 1];
        if (z > a) cnt[i] = wpre[z / kSlotWord] - wpre[a / kSlotWord];
    }
}

// The entries of the HBM tables into the coarse CSR, a wavefront per kEmitRun
// consecutive words (one lane per slot): the first word's row by binary
// search, the next ones by walking on.  A table spreads over as many
// wavefronts as it has slots (R-MAT scale 20's first coarse graph, one
// community holding a quarter of it: 0.09 ms, against 7.7 ms with a wavefront
// per row, and 6.4 ms more to count them that way).
constexpr int kEmitRun = 32;
__global__ void __launch_bounds__(kBlock)
coarse_emit_hbm_kernel(const int64_t* __restrict__ toff, const int* __restrict__ tkey,
                       const fx_t* __restrict__ tval, int64_t K, const int64_t* __restrict__ wpre, int64_t nwords,
                       const int64_t* __restrict__ noff, int64_t* __restrict__ ncol, int* __restrict__ ncol32,
                       double* __restrict__ nw_out)
{
    const int lane = threadIdx.x & 63;
    const int64_t nw = (int64_t)gridDim.x * (kBlock / 64);
    for (int64_t t = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); t * kEmitRun < nwords; t += nw) {
        const int64_t x0 = t * kEmitRun, x1 = x0 + kEmitRun < nwords ? x0 + kEmitRun : nwords;
        int64_t i = 0, r = K;              // toff[i] <= x0 * kSlotWord < toff[r]
        while (r - i > 1) {
            const int64_t mid = (i + r) / 2;
            if (toff[mid] <= x0 * kSlotWord) i = mid;
            else r = mid;
        }
        int64_t z = toff[i + 1], delta = noff[i] - wpre[toff[i] / kSlotWord];
        for (int64_t x = x0; x < x1; ++x) {
            while (z <= x * kSlotWord) {   // x < nwords: ends at a row with slots
                ++i;
                z = toff[i + 1];
                if (z > x * kSlotWord) delta = noff[i] - wpre[toff[i] / kSlotWord];
            }
            const int64_t s = x * kSlotWord + lane;
            const int c = tkey[s];
            const unsigned long long m = __ballot(c >= 0);
            if (c >= 0) {
                const int64_t p = delta + wpre[x] + __popcll(m & ((1ull << lane) - 1));
                ncol[p] = c;
                ncol32[p] = c;
                nw_out[p] = fx_to_double(tval[s]);
            }
        }
    }
}

// The compact entries of the LDS-aggregated rows into the coarse CSR.
__global__ void __launch_bounds__(kBlock)
coarse_emit_kernel(const int64_t* __restrict__ toff, int64_t K, const int64_t* __restrict__ noff,
                   int64_t* __restrict__ ncol, int* __restrict__ ncol32, double* __restrict__ nw_out,
                   const int64_t* __restrict__ cpos,
                   const int* __restrict__ ckey, const double* __restrict__ cw)
{
    const int lane = threadIdx.x & 63;
    const int64_t wid = (blockIdx.x * (int64_t)kBlock + threadIdx.x) >> 6;
    const int64_t nw = ((int64_t)gridDim.x * kBlock) >> 6;
    for (int64_t i = wid; i < K; i += nw) {
        if (toff[i + 1] != toff[i]) continue;   // uniform: an HBM row
        const int64_t pos = noff[i], n = noff[i + 1] - pos, c0 = cpos[i];
        for (int64_t r = lane; r < n; r += 64) {
            ncol[pos + r] = ckey[c0 + r];
            ncol32[pos + r] = ckey[c0 + r];
            nw_out[pos + r] = cw[c0 + r];
        }
    }
}

// ---------------------------------------------------------------------------
// Several graphs in one CSR: per-graph modularity, graph ids, vertex bases.
// ---------------------------------------------------------------------------
// Item = arcs [e0, e1) and vertices [v0, v1) of graph g; each workgroup sums
// its item exactly and adds the two sums to graph g's accumulators with
// integer atomics (order-free, so the result is exact and deterministic).
__global__ void __launch_bounds__(kBlock)
mod_seg_kernel(const SegItem* __restrict__ items, int64_t nitems, const int* __restrict__ src,
               const int* __restrict__ col, const double* __restrict__ w, const int* __restrict__ C,
               const fx_t* __restrict__ a, const double* __restrict__ twom_g, fx_t* __restrict__ acc,
               const unsigned char* __restrict__ act, fx_t* __restrict__ term)
{
    __shared__ fx_t red[kBlock / 64];
    for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x) {
        const SegItem s = items[it];
        if (act && !act[s.g]) continue;   // uniform: a graph that sat out kept its partition
        fx_t I = 0, T = 0;
        for (int64_t e = s.e0 + threadIdx.x; e < s.e1; e += kBlock)
            if (C[src[e]] == C[col[e]]) I += fx_from_double(w[e]);    // self arcs are internal
        const double tw = twom_g[s.g];
        for (int64_t i = s.v0 + threadIdx.x; i < s.v1; i += kBlock) {
            const double x = fx_to_double(a[i]) / tw;
            const fx_t t = fx_from_double(x * x);
            if (term) term[i] = t;
            T += t;
        }
        I = block_sum_fx(I, red);
        T = block_sum_fx(T, red);
        if (threadIdx.x == 0) {
            acc_add(acc + 2 * s.g, I);
            acc_add(acc + 2 * s.g + 1, T);
        }
    }
}

__global__ void __launch_bounds__(kBlock)
mod_seg_finalize_kernel(const fx_t* __restrict__ acc, const double* __restrict__ twom_g, int G,
                        double* __restrict__ q, const unsigned char* __restrict__ act,
                        const unsigned long long* __restrict__ moved)
{
    __shared__ unsigned long long red[kBlock / 64];
    for (int g = blockIdx.x * kBlock + threadIdx.x; g < G; g += gridDim.x * kBlock) {
        if (act && !act[g]) continue;     // q[g] keeps the value of its last evaluation
        const double tw = twom_g[g];
        q[g] = tw == 0 ? 0.0 : fx_to_double(acc[2 * g]) / tw - fx_to_double(acc[2 * g + 1]);
    }
    if (moved && blockIdx.x == 0) {   // uniform
        const unsigned long long t = sum_moved_slots(moved, red);
        if (threadIdx.x == 0) reinterpret_cast<unsigned long long*>(q)[G] = t;
    }
}

// out[g] = newid[vb[g]] (the scan total where vb[g] == nv), g = 0..G.
__global__ void __launch_bounds__(kBlock)
gather_bases_kernel(const int64_t* __restrict__ newid, const int64_t* __restrict__ total,
                    const int64_t* __restrict__ vb, int G, int64_t nv, int64_t* __restrict__ out)
{
    for (int g = blockIdx.x * kBlock + threadIdx.x; g <= G; g += gridDim.x * kBlock)
        out[g] = vb[g] < nv ? newid[vb[g]] : *total;
}

// out[g] = the exact sum of k over graph g's vertices; one workgroup per graph.
__global__ void __launch_bounds__(kBlock)
graph_sums_kernel(const fx_t* __restrict__ k, const int64_t* __restrict__ vb, int G, fx_t* __restrict__ out)
{
    __shared__ fx_t red[kBlock / 64];
    for (int g = blockIdx.x; g < G; g += gridDim.x) {
        fx_t t = 0;
        for (int64_t v = vb[g] + threadIdx.x; v < vb[g + 1]; v += kBlock) t += k[v];
        t = block_sum_fx(t, red);
        if (threadIdx.x == 0) out[g] = t;
    }
}

// gid[i] = g for i in [vb[g], vb[g+1]); one workgroup per graph.
__global__ void __launch_bounds__(kBlock)
fill_gid_kernel(const int64_t* __restrict__ vb, int G, int* __restrict__ gid)
{
    for (int g = blockIdx.x; g < G; g += gridDim.x)
        for (int64_t i = vb[g] + threadIdx.x; i < vb[g + 1]; i += kBlock) gid[i] = g;
}

}  // namespace

// ---------------------------------------------------------------------------
// Launch helpers
// ---------------------------------------------------------------------------
void launch_fill_i64(int64_t* p, int64_t val, int64_t n, hipStream_t s)
{
    if (n <= 0) return;
    fill_kernel<int64_t><<<grid_for(n, kBlock * 4), kBlock, 0, s>>>(p, val, n);
}

void launch_take_arcs(const ArcPiece* pieces, int64_t n, int64_t ne, int64_t nv, const int64_t* col, const double* w,
                      int* col32, WeightGrid* G, hipStream_t s)
{
    grid_init_kernel<<<1, 1, 0, s>>>(G);
    if (n > 0) take_arcs_kernel<<<grid_for(n, 1, 8192), kBlock, 0, s>>>(pieces, n, ne, nv, col, w, col32, G);
}

void launch_to_fixed(const double* w, int64_t* wq, int64_t ne, double scale, hipStream_t s)
{
    if (ne > 0) to_fixed_kernel<<<grid_for(ne, kBlock * 4), kBlock, 0, s>>>(w, wq, ne, scale);
}

void launch_iota_i64(int64_t* p, int64_t n, hipStream_t s)
{
    if (n <= 0) return;
    iota_kernel<<<grid_for(n, kBlock * 4), kBlock, 0, s>>>(p, n);
}

void launch_fill_i32(int32_t* p, int32_t val, int64_t n, hipStream_t s)
{
    if (n <= 0) return;
    fill_kernel<int32_t><<<grid_for(n, kBlock * 4), kBlock, 0, s>>>(p, val, n);
}

void launch_fill_fx(fx_t* p, int64_t n, hipStream_t s)
{
    if (n <= 0) return;
    fill_kernel<fx_t><<<grid_for(n, kBlock * 4), kBlock, 0, s>>>(p, (fx_t)0, n);
}

void launch_vertex_weights(const int64_t* off, const double* w, int64_t ne, fx_t* k, double* kd, int64_t nv,
                           PhaseOut* out, fx_t* part, int* src, hipStream_t s)
{
    phase_init_kernel<<<1, 1, 0, s>>>(out);
    if (nv <= 0) return;
    launch_fill_fx(k, nv, s);
    if (ne > 0)
        row_sums_kernel<<<grid_for(ne, kSumTile, 8192), kBlock, 0, s>>>(off, w, nv, ne, k, src, &out->grid);
    const unsigned g = grid_for(nv, kBlock, kPartBlocks);
    round_kernel<<<g, kBlock, 0, s>>>(k, kd, nv, &out->maxk, part);
    sum_partials_kernel<<<1, kBlock, 0, s>>>(part, (int)g, &out->twom);
}

void launch_fx_round(const fx_t* x, double* out, int64_t n, hipStream_t s)
{
    if (n > 0) fx_round_kernel<<<grid_for(n, kBlock), kBlock, 0, s>>>(x, out, n);
}

void launch_singleton(int64_t* C, int64_t* Cn, int* C32, fx_t* a, const fx_t* k, int64_t nv,
                      hipStream_t s)
{
    if (nv <= 0) return;
    singleton_kernel<<<grid_for(nv, kBlock), kBlock, 0, s>>>(C, Cn, C32, a, k, nv);
}


void launch_widen_ids(const int* col32, int64_t* col, int64_t n, hipStream_t s)
{
    if (n <= 0) return;
    widen_kernel<<<grid_for(n, kBlock), kBlock, 0, s>>>(col32, col, n);
}

void launch_modularity(const int* src, const int* col, const double* w, const int* C,
                       int64_t ne, const fx_t* a, int64_t nv, double twom_d, fx_t* part, double* q,
                       hipStream_t s, fx_t* term, fx_t* acc, bool ident)
{
    const int64_t tiles = (ne + (int64_t)kBlock * kModUnroll - 1) / ((int64_t)kBlock * kModUnroll);
    const int64_t need = tiles > (nv + kBlock - 1) / kBlock ? tiles : (nv + kBlock - 1) / kBlock;
    const unsigned g = grid_for(need, 1, kPartBlocks);
    if (ident) mod_kernel<true><<<g, kBlock, 0, s>>>(src, col, w, C, ne, a, nv, twom_d, part, term);
    else mod_kernel<false><<<g, kBlock, 0, s>>>(src, col, w, C, ne, a, nv, twom_d, part, term);
    mod_finalize_kernel<<<1, kBlock, 0, s>>>(part, (int)g, twom_d, q, acc);
}

void launch_modularity_rows(const int64_t* off, const int* col, const double* w, const int* C, int64_t v0,
                            int64_t v1, int64_t arcs, fx_t* acc, hipStream_t s)
{
    if (v1 > v0 && arcs > 0)
        mod_rows_kernel<<<grid_for(arcs, (int64_t)kBlock * kModRun, 8192), kBlock, 0, s>>>(off, col, w, C, v0, v1,
                                                                                            acc);
}

void launch_modularity_terms(const fx_t* a, int64_t nv, double twom_d, fx_t* acc, double* q, hipStream_t s,
                             fx_t* term)
{
    if (nv > 0) mod_terms_kernel<<<grid_for(nv, kBlock, kPartBlocks), kBlock, 0, s>>>(a, nv, twom_d, acc, term);
    mod_acc_finish_kernel<<<1, 64, 0, s>>>(acc, twom_d, q);
}

void launch_sym_hash(const int* src, const int* col, const double* w, int64_t ne, unsigned long long* part,
                     unsigned long long* out, hipStream_t s)
{
    static_assert(4 * sizeof(unsigned long long) == 2 * sizeof(fx_t), "kPartBlocks workgroups' sums fit the partials");
    const unsigned g = grid_for(ne, kBlock, kPartBlocks);
    sym_hash_kernel<<<g, kBlock, 0, s>>>(src, col, w, ne, part);
    sym_sum_kernel<<<1, kBlock, 0, s>>>(part, (int)g, out);
}

void launch_mod_delta(int b, int64_t v0, int64_t v1, const int64_t* Cn, const int* C32, const int* col,
                      const double* w, const fx_t* a, double twom_d, const ModDelta& D, hipStream_t s)
{
    mod_delta_kernel<<<512, kBlock, 0, s>>>(b, v0, v1, Cn, C32, col, w, a, twom_d, D);
}

void launch_mod_finish_graphs(const ModDelta& D, int nb, int G, double* q, const unsigned char* act,
                              hipStream_t s)
{
    mod_finish_graphs_kernel<<<grid_for(G, kBlock), kBlock, 0, s>>>(D, nb, G, q, act);
}

void launch_mod_finish(const ModDelta& D, int nb, double twom_d, double* q, hipStream_t s)
{
    mod_finish_kernel<<<1, kBlock, 0, s>>>(D, nb, twom_d, q);
}

size_t scan_temp_bytes(int64_t n)
{
    size_t bytes = 0;
    int64_t m = n;
    while (m > kScanTile) {
        m = (m + kScanTile - 1) / kScanTile;
        bytes += (size_t)m * sizeof(int64_t);
    }
    return bytes + 64;
}

static void scan_rows(const int64_t* in, int64_t* out, int64_t n, int rows, int64_t stride, int64_t* total,
                      int64_t* totals, void* temp, hipStream_t s)
{
    const int64_t tiles = (n + kScanTile - 1) / kScanTile;
    const dim3 grid((unsigned)tiles, (unsigned)rows);
    if (tiles == 1) {
        scan_tile_apply_kernel<<<grid, kBlock, 0, s>>>(in, out, n, nullptr, total, stride, totals);
        return;
    }
    int64_t* sums = reinterpret_cast<int64_t*>(temp);
    void* rest = sums + tiles * rows;
    scan_tile_sums_kernel<<<grid, kBlock, 0, s>>>(in, n, sums, stride);
    scan_rows(sums, sums, tiles, rows, tiles, nullptr, nullptr, rest, s);
    scan_tile_apply_kernel<<<grid, kBlock, 0, s>>>(in, out, n, sums, total, stride, totals);
}

void launch_exclusive_scan(const int64_t* in, int64_t* out, int64_t n, int64_t* total,
                           void* temp, hipStream_t s)
{
    if (n <= 0) {
        if (total) launch_fill_i64(total, 0, 1, s);
        return;
    }
    scan_rows(in, out, n, 1, 0, total, nullptr, temp, s);
}

void launch_exclusive_scans(int64_t* x, int64_t n, int rows, int64_t stride, int64_t* totals, void* temp,
                            hipStream_t s)
{
    if (n > 0) scan_rows(x, x, n, rows, stride, x + n, totals, temp, s);
}

void launch_mark_communities(const int64_t* C, int64_t nv, int64_t* flag, hipStream_t s,
                             const int* gid, const unsigned char* keep)
{
    launch_fill_i64(flag, 0, nv, s);
    if (nv > 0) mark_kernel<<<grid_for(nv, kBlock), kBlock, 0, s>>>(C, nv, flag, gid, keep);
}

void launch_update_clustering(int64_t* clus, int64_t n0, const int64_t* C, const int64_t* newid,
                              hipStream_t s, const int* gid0, const unsigned char* keep)
{
    if (n0 > 0) clustering_kernel<<<grid_for(n0, kBlock), kBlock, 0, s>>>(clus, n0, C, newid, gid0, keep);
}

void launch_widen_local(const ArcPiece* pieces, int64_t n, const uint16_t* local, int* col32, hipStream_t s)
{
    if (n > 0) widen_local_kernel<<<grid_for(n, 1, 16384), kBlock, 0, s>>>(pieces, n, local, col32);
}

void launch_local_ids(const int64_t* clus, int64_t n0, const int* gid0, const int64_t* base, int64_t* out,
                      hipStream_t s)
{
    if (n0 > 0) local_ids_kernel<<<grid_for(n0, kBlock), kBlock, 0, s>>>(clus, n0, gid0, base, out);
}

void launch_member_counts(const int64_t* C, const int64_t* newid, const int64_t* off, int64_t nv, int* cid,
                          int64_t* cnt, int64_t* arcs, hipStream_t s, const int* gid, const unsigned char* keep)
{
    if (nv > 0)
        member_counts_kernel<<<grid_for(nv, kBlock), kBlock, 0, s>>>(C, newid, off, nv, cid, cnt, arcs, gid, keep);
}

void launch_coarse_sizes(const int64_t* arcs, const int64_t* cnt, int64_t K, const CoarseRows& R, hipStream_t s)
{
    if (K > 0)
        coarse_sizes_kernel<<<grid_for(K, kBlock), kBlock, 0, s>>>(arcs, cnt, K, R.ml, R.mh, R.toff, R.cpos, R.mid,
                                                                   R.nmid);
}

void launch_member_scatter(const int* cid, const int64_t* off, int64_t nv, const CoarseRows& R, int64_t ML,
                           unsigned long long* mfill, int* members, int64_t* hd, hipStream_t s)
{
    if (nv > 0)
        member_scatter_kernel<<<grid_for(nv, kBlock), kBlock, 0, s>>>(cid, off, nv, R.ml, R.mh, ML, R.toff, mfill,
                                                                       members, hd);
}

void launch_coarse_lds(const int64_t* arcs, const CoarseRows& R, const int* members, const int64_t* off,
                       const int* col, const double* w, const int* cid, int64_t K, int* ckey, double* cw,
                       int64_t* cnt, hipStream_t s)
{
    if (K <= 0) return;
    coarse_wave_kernel<<<grid_for(K, kBlock / 64), kBlock, 0, s>>>(arcs, R.ml, members, off, col, w, cid, K, R.cpos,
                                                                   ckey, cw, cnt);
    coarse_lds_kernel<<<grid_for(K, 1, 2048), kBlock, 0, s>>>(arcs, R.ml, members, off, col, w, cid, K, R.mid,
                                                              R.nmid, R.cpos, ckey, cw, cnt);
}

void launch_coarse_insert(const int64_t* hpre, int64_t n, int64_t max_arcs, const int* members, const int* cid,
                          const int64_t* off, const int* col, const double* w, const int64_t* toff, int* tkey,
                          fx_t* tval, hipStream_t s)
{
    if (n > 0)
        coarse_insert_kernel<<<grid_for(max_arcs, kInsTile, 16384), kBlock, 0, s>>>(hpre, n, members, cid, off, col, w,
                                                                                   toff, tkey, tval);
}

void launch_modularity_seg(const SegItem* items, int64_t nitems, const int* src, const int* col,
                           const double* w, const int* C, const fx_t* a, const double* twom_g, int G,
                           fx_t* acc, double* q, hipStream_t s, const unsigned char* act, fx_t* term,
                           const unsigned long long* moved)
{
    if (G <= 0) return;
    launch_fill_fx(acc, 2 * (int64_t)G, s);
    if (nitems > 0)
        mod_seg_kernel<<<grid_for(nitems, 1, 8192), kBlock, 0, s>>>(items, nitems, src, col, w, C, a,
                                                                    twom_g, acc, act, term);
    mod_seg_finalize_kernel<<<grid_for(G, kBlock), kBlock, 0, s>>>(acc, twom_g, G, q, act, moved);
}

void launch_graph_sums(const fx_t* k, const int64_t* vb, int G, fx_t* out, hipStream_t s)
{
    if (G > 0) graph_sums_kernel<<<grid_for(G, 1, 8192), kBlock, 0, s>>>(k, vb, G, out);
}

void launch_gather_bases(const int64_t* newid, const int64_t* total, const int64_t* vb, int G, int64_t nv,
                         int64_t* out, hipStream_t s)
{
    gather_bases_kernel<<<grid_for(G + 1, kBlock), kBlock, 0, s>>>(newid, total, vb, G, nv, out);
}

void launch_fill_gid(const int64_t* vb, int G, int* gid, hipStream_t s)
{
    if (G > 0) fill_gid_kernel<<<grid_for(G, 1, 8192), kBlock, 0, s>>>(vb, G, gid);
}

void launch_slot_words(const int* tkey, int64_t nwords, int64_t* wcnt, hipStream_t s)
{
    if (nwords > 0)
        slot_words_kernel<<<grid_for(nwords, kBlock / 64, 16384), kBlock, 0, s>>>(tkey, nwords, wcnt);
}

void launch_coarse_count(const int64_t* toff, const int64_t* wpre, int64_t K, int64_t* cnt, hipStream_t s)
{
    if (K > 0) coarse_count_kernel<<<grid_for(K, kBlock), kBlock, 0, s>>>(toff, wpre, K, cnt);
}

void launch_coarse_emit(const int64_t* toff, int64_t K, const int64_t* noff, int64_t* ncol, int* ncol32, double* nw,
                        const int64_t* cpos, const int* ckey, const double* cw, hipStream_t s)
{
    if (K > 0)
        coarse_emit_kernel<<<grid_for(K, kBlock / 64), kBlock, 0, s>>>(toff, K, noff, ncol, ncol32, nw, cpos, ckey,
                                                                       cw);
}

void launch_coarse_emit_hbm(const int64_t* toff, const int* tkey, const fx_t* tval, int64_t K, const int64_t* wpre,
                            int64_t nwords, const int64_t* noff, int64_t* ncol, int* ncol32, double* nw, hipStream_t s)
{
    if (nwords > 0)
        coarse_emit_hbm_kernel<<<grid_for(nwords, kEmitRun * (kBlock / 64)), kBlock, 0, s>>>(
            toff, tkey, tval, K, wpre, nwords, noff, ncol, ncol32, nw);
}

}  // namespace nido
