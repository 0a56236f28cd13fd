// Morton (Z-order) sort of particles on the GPU, with the exact order of
// the reference's starsh_particles_zsort_inplace
// (src/applications/particles.c:1090-1221 of ecrc/stars-h 0.3.1).
//
// The reference scales every coordinate to u = (x - min)/(max - min) *
// UINT32_MAX (truncated to uint32) and sorts by a recursive binary
// partition that visits, from bit 31 down to bit 0, dimensions ndim-1 down
// to 0, moving 0-bit points to the front in order and 1-bit points to the
// back in reverse order.  The result is the order of the interleaved key
//   key = sum_{b, d} bit b of u_d at position b*ndim + d,
// with points of equal key in their original order when the key has an
// even number of 1 bits and in reverse order when odd (each 1 bit reverses
// them once).  Here a stable LSD radix sort on the Morton key, 8 bits per
// pass, leaves equal keys in their original order, and the gather reverses
// the groups of odd parity:
//   zs_minmax_*   per-dimension min and max (exact, any reduction order);
//   zs_key        the key words of every point;
//   zs_load       the word being sorted by, in the current order;
//   zs_hist       per-tile digit counts;  zs_scan  offsets within a digit;
//   zs_scatter    stable scatter of (word, index): each tile ranks its points
//                 by digit in their order, with wave ballots for ranks
//                 inside a wave;
//   zs_gather     groups of equal keys, permutation and coordinates.
//
// What bounds it: launches and the scattered writes of a pass.  A million
// points in 3D (12 passes) take 0.50 ms on MI355X; with one workgroup
// scanning all digit counts of a pass (432 of the 510 us of a pass), all key
// words moved in every pass and three passes for the tie-break it was 7.6
// ms.
#include <stdio.h>
#include <algorithm>
#include <utility>
#include "hip_common.h"

namespace {

constexpr int ZT = 256;          // threads per block
constexpr int ZI = 4;            // points per thread per tile
constexpr int TILE = ZT*ZI;      // points per tile
constexpr int NDIG = 256;        // 8-bit digits

__global__ __launch_bounds__(ZT) void zs_minmax_partial(const double *x,
        int64_t n, int ndim, double *part)
{
    // part[(b * ndim + d) * 2 + {0, 1}] = min, max of block b
    __shared__ double smin[ZT], smax[ZT];
    for(int d = 0; d < ndim; d++)
    {
        double lo = INFINITY, hi = -INFINITY;
        for(int64_t i = (int64_t)blockIdx.x*ZT+threadIdx.x; i < n;
                i += (int64_t)gridDim.x*ZT)
        {
            const double v = x[(int64_t)d*n+i];
            lo = fmin(lo, v);
            hi = fmax(hi, v);
        }
        smin[threadIdx.x] = lo;
        smax[threadIdx.x] = hi;
        __syncthreads();
        for(int o = ZT/2; o > 0; o >>= 1)
        {
            if(threadIdx.x < o)
            {
                smin[threadIdx.x] = fmin(smin[threadIdx.x],
                        smin[threadIdx.x+o]);
                smax[threadIdx.x] = fmax(smax[threadIdx.x],
                        smax[threadIdx.x+o]);
            }
            __syncthreads();
        }
        if(threadIdx.x == 0)
        {
            part[((int64_t)blockIdx.x*ndim+d)*2] = smin[0];
            part[((int64_t)blockIdx.x*ndim+d)*2+1] = smax[0];
        }
        __syncthreads();
    }
}

// One block per dimension: mm[d] = min, mm[ndim + d] = max.
__global__ __launch_bounds__(ZT) void zs_minmax_final(const double *part,
        int nb, int ndim, double *mm)
{
    __shared__ double smin[ZT/64], smax[ZT/64];
    const int d = blockIdx.x;
    double lo = INFINITY, hi = -INFINITY;
    for(int b = threadIdx.x; b < nb; b += ZT)
    {
        lo = fmin(lo, part[((int64_t)b*ndim+d)*2]);
        hi = fmax(hi, part[((int64_t)b*ndim+d)*2+1]);
    }
    for(int o = 32; o > 0; o >>= 1)
    {
        lo = fmin(lo, __shfl_xor(lo, o, 64));
        hi = fmax(hi, __shfl_xor(hi, o, 64));
    }
    if((threadIdx.x & 63) == 0)
    {
        smin[threadIdx.x >> 6] = lo;
        smax[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if(threadIdx.x == 0)
    {
        for(int w = 1; w < ZT/64; w++)
        {
            lo = fmin(lo, smin[w]);
            hi = fmax(hi, smax[w]);
        }
        mm[d] = lo;
        mm[ndim+d] = hi;
    }
}

// Key words of point i (SoA, NDIM words of n, least significant first).
template <int NDIM>
__global__ __launch_bounds__(ZT) void zs_key(const double *x, int64_t n,
        const double *mm, uint32_t *key, uint32_t *idx)
{
    const int64_t i = (int64_t)blockIdx.x*ZT+threadIdx.x;
    if(i >= n)
        return;
    uint32_t u[NDIM];
#pragma unroll
    for(int d = 0; d < NDIM; d++)
    {
        const double lo = mm[d], range = mm[NDIM+d]-lo;
        // the reference's expression: (x - min)/range*UINT32_MAX, then
        // conversion to uint32 (truncation)
        const double v = (x[(int64_t)d*n+i]-lo)/range*4294967295.0;
        u[d] = (uint32_t)v;
    }
    // bit b of u_d goes to key bit b*NDIM + d; key word w holds bits
    // 32w .. 32w+31
    uint32_t w[NDIM];
#pragma unroll
    for(int q = 0; q < NDIM; q++)
        w[q] = 0;
#pragma unroll
    for(int b = 0; b < 32; b++)
#pragma unroll
        for(int d = 0; d < NDIM; d++)
        {
            const int pos = b*NDIM+d;
            w[pos >> 5] |= ((u[d] >> b) & 1u) << (pos & 31);
        }
#pragma unroll
    for(int q = 0; q < NDIM; q++)
        key[(int64_t)q*n+i] = w[q];
    idx[i] = (uint32_t)i;
}

// wk[i] = the word of the point at place i.
__global__ __launch_bounds__(ZT) void zs_load(const uint32_t *key, int64_t n,
        const uint32_t *idx, uint32_t *wk)
{
    const int64_t i = (int64_t)blockIdx.x*ZT+threadIdx.x;
    if(i < n)
        wk[i] = key[min((int64_t)idx[i], n-1)];
}

__device__ inline uint32_t digit_of(const uint32_t *wk, int shift, int64_t i)
{
    return (wk[i] >> shift) & (NDIG-1);
}

__global__ __launch_bounds__(ZT) void zs_hist(const uint32_t *wk, int64_t n,
        int shift, uint32_t *hist, int ntile)
{
    __shared__ uint32_t cnt[NDIG];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const int64_t t0 = (int64_t)blockIdx.x*TILE;
    for(int r = 0; r < ZI; r++)
    {
        const int64_t i = t0+r*ZT+threadIdx.x;
        if(i < n)
            atomicAdd(&cnt[digit_of(wk, shift, i)], 1u);
    }
    __syncthreads();
    hist[(int64_t)threadIdx.x*ntile+blockIdx.x] = cnt[threadIdx.x];
}

// Exclusive scan over a block of ZT threads; *total is the sum.
__device__ inline uint32_t block_scan(uint32_t v, uint32_t *wsum,
        uint32_t *total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
    for(int o = 1; o < 64; o <<= 1)
    {
        const uint32_t y = __shfl_up(x, o, 64);
        if(lane >= o)
            x += y;
    }
    if(lane == 63)
        wsum[wave] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for(int w = 0; w < ZT/64; w++)
    {
        before += w < wave ? wsum[w] : 0;
        all += wsum[w];
    }
    __syncthreads();
    *total = all;
    return before+x-v;
}

// One block per digit: exclusive scan of its ntile counts in place, their
// sum to total[digit].
__global__ __launch_bounds__(ZT) void zs_scan(uint32_t *hist, int ntile,
        uint32_t *total)
{
    __shared__ uint32_t wsum[ZT/64];
    uint32_t *v = hist+(int64_t)blockIdx.x*ntile;
    uint32_t carry = 0;
    for(int c0 = 0; c0 < ntile; c0 += ZT)
    {
        const int i = c0+threadIdx.x;
        uint32_t sum;
        const uint32_t x = block_scan(i < ntile ? v[i] : 0, wsum, &sum);
        if(i < ntile)
            v[i] = carry+x;
        carry += sum;
    }
    if(threadIdx.x == 0)
        total[blockIdx.x] = carry;
}

__global__ __launch_bounds__(ZT) void zs_scatter(const uint32_t *wk,
        const uint32_t *idx, uint32_t *wk2, uint32_t *idx2, int64_t n,
        int shift, const uint32_t *off, const uint32_t *total, int ntile)
{
    __shared__ uint32_t base[NDIG];      // tile offset + points placed so far
    __shared__ uint32_t wcnt[ZT/64][NDIG];
    __shared__ uint32_t wsum[ZT/64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // digit offsets: every block scans the 256 totals for itself
    uint32_t all;
    base[threadIdx.x] = block_scan(total[threadIdx.x], wsum, &all)+
        off[(int64_t)threadIdx.x*ntile+blockIdx.x];
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64-lane));
    const int64_t t0 = (int64_t)blockIdx.x*TILE;
    for(int r = 0; r < ZI; r++)
    {
        for(int w = 0; w < ZT/64; w++)
            wcnt[w][threadIdx.x] = 0;
        __syncthreads();
        // points of this round, in order: thread t takes t0 + r*ZT + t
        const int64_t i = t0+r*ZT+threadIdx.x;
        const bool valid = i < n;
        const uint32_t word = valid ? wk[i] : 0;
        const uint32_t dg = (word >> shift) & (NDIG-1);
        // lanes of this wave with the same digit
        uint64_t peers = __ballot(valid);
        for(int b = 0; b < 8; b++)
        {
            const uint64_t m = __ballot(((dg >> b) & 1u) != 0);
            peers &= ((dg >> b) & 1u) ? m : ~m;
        }
        const uint32_t before = (uint32_t)__popcll(peers & lt);
        if(valid && before == 0)
            wcnt[wave][dg] = (uint32_t)__popcll(peers);
        __syncthreads();
        if(valid)
        {
            uint32_t pos = base[dg]+before;
            for(int w = 0; w < wave; w++)
                pos += wcnt[w][dg];
            // pos < n by construction (offsets of a full histogram); the
            // test keeps a wrong offset from writing out of bounds
            if(pos >= (uint64_t)n)
                pos = (uint32_t)(n-1);
            wk2[pos] = word;
            idx2[pos] = idx[i];
        }
        __syncthreads();
        uint32_t add = 0;
        for(int w = 0; w < ZT/64; w++)
            add += wcnt[w][threadIdx.x];
        base[threadIdx.x] += add;
        __syncthreads();
    }
}

// -1, 0, 1 as the key of point a is below, equal to or above that of b.
__device__ inline int key_cmp(const uint32_t *key, int64_t n, int ndim,
        uint32_t a, uint32_t b)
{
    for(int q = ndim-1; q >= 0; q--)
    {
        const uint32_t ka = key[(int64_t)q*n+a], kb = key[(int64_t)q*n+b];
        if(ka != kb)
            return ka < kb ? -1 : 1;
    }
    return 0;
}

// The point of place i: idx[i], or, in a group of equal keys (places lo ..
// hi-1, found by bisection) with an odd number of 1 bits, idx[lo+hi-1-i].
// wk: the most significant key words in order.
__global__ __launch_bounds__(ZT) void zs_gather(const double *x, int64_t n,
        int ndim, const uint32_t *key, const uint32_t *wk,
        const uint32_t *idx, double *y, int64_t *order)
{
    const int64_t i = (int64_t)blockIdx.x*ZT+threadIdx.x;
    if(i >= n)
        return;
    uint32_t j = idx[i];
    const bool tied = (i > 0 && wk[i-1] == wk[i] &&
            key_cmp(key, n, ndim, idx[i-1], j) == 0) ||
        (i+1 < n && wk[i+1] == wk[i] &&
         key_cmp(key, n, ndim, idx[i+1], j) == 0);
    if(tied)
    {
        int ones = 0;
        for(int q = 0; q < ndim; q++)
            ones += __popc(key[(int64_t)q*n+j]);
        if(ones & 1)
        {
            int64_t lo = 0, hi = i;         // first place not below j's key
            while(lo < hi)
            {
                const int64_t mid = (lo+hi)/2;
                if(key_cmp(key, n, ndim, idx[mid], j) < 0)
                    lo = mid+1;
                else
                    hi = mid;
            }
            int64_t first = i+1, last = n;  // first place above it
            while(first < last)
            {
                const int64_t mid = (first+last)/2;
                if(key_cmp(key, n, ndim, idx[mid], j) <= 0)
                    first = mid+1;
                else
                    last = mid;
            }
            j = idx[lo+first-1-i];
        }
    }
    j = j < (uint64_t)n ? j : 0;
    for(int d = 0; d < ndim; d++)
        y[(int64_t)d*n+i] = x[(int64_t)d*n+j];
    if(order)
        order[i] = j;
}

} // namespace

// Sorts n points (SoA, ndim x n, at d_x) into Morton order: d_y gets the
// permuted coordinates, d_order (optional) the permutation (d_y[., i] =
// d_x[., d_order[i]]).  d_x and d_y must not overlap.
extern "C" int starsh_hip_zsort(const double *d_x, int64_t n, int ndim,
        double *d_y, int64_t *d_order)
{
    if(n < 0 || n > 0x7fffffff || ndim < 1 || ndim > 4 ||
            (n > 0 && (d_x == nullptr || d_y == nullptr)))
        return STARSH_WRONG_PARAMETER;
    if(n == 0)
        return STARSH_SUCCESS;
    int info = starsh_hip_init(0);
    if(info != STARSH_SUCCESS)
        return info;
    hipStream_t s = starsh_hip_stream();
    const int ntile = (int)((n+TILE-1)/TILE);
    const int nbmm = (int)std::min<int64_t>((n+ZT-1)/ZT, 1024);
    // scratch: min/max partials, key words, the sorted word and the indices
    // twice, histogram and digit totals
    size_t bytes = sizeof(double)*((size_t)nbmm*ndim*2+2*ndim)+
        sizeof(uint32_t)*((size_t)n*ndim+4*(size_t)n+(size_t)NDIG*ntile+
                NDIG);
    char *buf = nullptr;
    HIP_TRY(hipMallocAsync((void **)&buf, bytes, s));
    double *part = (double *)buf;
    double *mm = part+(size_t)nbmm*ndim*2;
    uint32_t *key = (uint32_t *)(mm+2*ndim);
    uint32_t *wk = key+(size_t)n*ndim;
    uint32_t *wk2 = wk+n;
    uint32_t *idx = wk2+n;
    uint32_t *idx2 = idx+n;
    uint32_t *hist = idx2+n;
    uint32_t *total = hist+(size_t)NDIG*ntile;
    const unsigned nb = (unsigned)((n+ZT-1)/ZT);
    hipLaunchKernelGGL(zs_minmax_partial, dim3(nbmm), dim3(ZT), 0, s, d_x, n,
            ndim, part);
    hipLaunchKernelGGL(zs_minmax_final, dim3(ndim), dim3(ZT), 0, s, part,
            nbmm, ndim, mm);
    switch(ndim)
    {
        case 1: hipLaunchKernelGGL(zs_key<1>, dim3(nb), dim3(ZT), 0, s, d_x,
                    n, mm, key, idx); break;
        case 2: hipLaunchKernelGGL(zs_key<2>, dim3(nb), dim3(ZT), 0, s, d_x,
                    n, mm, key, idx); break;
        case 3: hipLaunchKernelGGL(zs_key<3>, dim3(nb), dim3(ZT), 0, s, d_x,
                    n, mm, key, idx); break;
        default: hipLaunchKernelGGL(zs_key<4>, dim3(nb), dim3(ZT), 0, s, d_x,
                    n, mm, key, idx); break;
    }
    for(int word = 0; word < ndim; word++)
    {
        hipLaunchKernelGGL(zs_load, dim3(nb), dim3(ZT), 0, s,
                key+(size_t)word*n, n, idx, wk);
        for(int shift = 0; shift < 32; shift += 8)
        {
            hipLaunchKernelGGL(zs_hist, dim3(ntile), dim3(ZT), 0, s, wk, n,
                    shift, hist, ntile);
            hipLaunchKernelGGL(zs_scan, dim3(NDIG), dim3(ZT), 0, s, hist,
                    ntile, total);
            hipLaunchKernelGGL(zs_scatter, dim3(ntile), dim3(ZT), 0, s, wk,
                    idx, wk2, idx2, n, shift, hist, total, ntile);
            std::swap(wk, wk2);
            std::swap(idx, idx2);
        }
    }
    hipLaunchKernelGGL(zs_gather, dim3(nb), dim3(ZT), 0, s, d_x, n, ndim,
            key, wk, idx, d_y, d_order);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipFreeAsync(buf, s));
    HIP_TRY(hipStreamSynchronize(s));
    return STARSH_SUCCESS;
}
