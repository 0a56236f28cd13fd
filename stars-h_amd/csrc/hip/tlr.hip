// Product of a compressed (tile low-rank) matrix with a dense block of
// vectors on the GPU, Y = alpha * M * X + beta * Y, and the vector kernels
// of conjugate gradients.  Follows src/backends/sequential/blrm/dmml.c:16-145
// of ecrc/stars-h 0.3.1: every far-field tile (i, j) adds U (V^T X_j) to Y_i
// and, in a symmetric format with i != j, V (U^T X_i) to Y_j; near-field
// tiles add D X_j (and D^T X_i).
//
// Two launches, both deterministic (no atomics):
//  1. one workgroup per 32 columns of a factor: the coefficients T = V^T X_j
//     and, for a tile with a twin (symmetric format, i != j), T' = U^T X_i;
//  2. one workgroup per strip of 64, 32 or 16 rows of one block row: the sum
//     of all contributions to those rows (U T, V T', D X_j, D^T X_i) in a
//     fixed order: wave w takes entries w, w+4, ... (wide ones come in
//     pieces) and the four partial sums are added in LDS in wave order.
// With one right-hand side a lane multiplies its own values; with more, up
// to 16 at a time go through FP64 MFMA (the columns past nrhs are zeros).
//
// Rounding: an MFMA adds its products to the accumulator one by one, so a
// long chain of them loses what a lane's short one kept.  Chains end after 16
// products and go to a sum of their own.  Relative errors against long double,
// for chains as long as a wave's share, now, and with a workgroup per tile and
// four right-hand sides at a time:
//   N=2500, tile 250, rank 30, 4 rhs            4.2, 2.7, 2.3 e-16
//   N=16000, tile 1000, rank 60, 16 rhs         7.2, 3.0, 2.6 e-16
//   N=30000, tile 1700, dense tiles, 10 rhs     7.2, 2.5, 13.6 e-16
//   N=64000, tile 1600, rank 31, 1 rhs          3.1, 2.7, 2.7 e-16
// Chains of 8 (2.3 and 2.7 e-16 for the first two) spill: 20-30% slower.
//
// What bounds it: memory; every factor is read twice, every dense tile once.
// A kernel that only reads runs at 6.0-6.2 TB/s here, 7.0 below 268 MB, which
// the cache in front of the memory holds; the coefficients of C2's operator
// (N=64000, tile 1600, 431 MB) run at 5.8, its rows at 6.3.  Measured on
// MI355X, before and after (one workgroup per tile forming U^T X and then
// V (U^T X) row by row, and strips of 64 rows, dense tiles one column at a
// time, right-hand sides in groups of four that each re-read everything):
//   N=2500, tile 250, 1 rhs (launch-bound)                  27.7 -> 10.7 us
//   N=64000, tile 1600, ranks 8-31, 1 rhs, 358 MB, read
//     twice                                              129-146 -> 116-122 us
//   the same with ranks to 133, 1566 MB                       578 -> 500 us
//   C2's operator (2D sqexp, 431 MB), 1 rhs               149-152 -> 141 us
//   N=30000, tile 1700, nonsymmetric, ranks to 90, 12 dense
//     tiles, 10 rhs, 812 MB                                 4470 -> 225 us
//   CG iteration, N=10000, tile 1000, 10 dense tiles         610 -> 72 us
// Reading U once for U^T X and keeping V (U^T X) (1.5 reads instead of 2)
// needs a workgroup per tile: 100 + 49 us for C2's operator against 74 + 67.
#include <stdio.h>
#include "hip_common.h"
#include "tlr.h"

typedef double double4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int RHS = 16;         // right-hand sides per group

// With more strips of 64 rows than this, one right-hand side goes through
// tlr_rows1_kernel.  tlr_rows_kernel<4, true> has more loads in flight but
// takes 154 registers, three workgroups per CU, 768 on the chip: 1000 strips
// (C2's operator, 431 MB) left a second round nearly empty, 150 us for the
// product against 141 with a lane per row (76 registers, six workgroups);
// 358 MB 117.9 against 116.3, 700 MB 227.4 against 227.1.  Within one round it
// wins: 563 strips 41.9 against 44.5 us, 625 46.2 against 46.9, 704 55.9
// against 56.5.
constexpr int ROWS1_STRIPS = 768;

// Sums of one 16 x 16 fragment over its k: four MFMA steps' worth of a lane's
// values f (row lane%16 of op(F)) times b.  With one right-hand side a lane
// adds up its own products (v[0]; summed over the four lane groups at the
// end), with more the MFMA does (row lane/16 + 4 v, column lane%16).
template <bool ONE>
struct Acc
{
    double4_t v = {0.0, 0.0, 0.0, 0.0};
    // adds another's sums and clears them
    __device__ inline void take(Acc &o)
    {
        if constexpr(ONE)
            v[0] += o.v[0];
        else
            v += o.v;
        o.v = double4_t{0.0, 0.0, 0.0, 0.0};
    }
    __device__ inline void add(double f, double b)
    {
        if constexpr(ONE)
            v[0] = fma(f, b, v[0]);
        else
            v = __builtin_amdgcn_mfma_f64_16x16x4f64(f, b, v, 0, 0, 0);
    }
    __device__ inline void close()
    {
        if constexpr(ONE)
        {
            v[0] += __shfl_xor(v[0], 16, 64);
            v[0] += __shfl_xor(v[0], 32, 64);
        }
    }
    // values per lane and the row of value q
    static constexpr int N = ONE ? 1 : 4;
    static __device__ inline int row(int q, int lane)
    {
        return ONE ? lane & 15 : (lane >> 4)+4*q;
    }
};

// S = F^T x for 32 columns of a factor F (len rows), one right-hand side: a
// lane takes a row of a 64-row chunk (512 contiguous bytes of a column per
// load), the chunks are striped over the four waves, and a wave's sums over
// its lanes come from one recursive halving of all its columns.  (The MFMA
// operand layout below, 32 bytes of 16 columns per row group, read the short
// factors of a 64000-row operator, 16 columns of 1600 rows, at 2.7 TB/s.)
__global__ __launch_bounds__(256) void tlr_coef1_kernel(const tlr_unit *units,
        const double *fac, const double *x, double *tmp)
{
    constexpr int C = 32;
    __shared__ double part[4][C];
    const tlr_unit u = units[blockIdx.x];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const double *F = fac+u.f_off, *X = x+u.x_off;
    double s[C];
#pragma unroll
    for(int c = 0; c < C; c++)
        s[c] = 0.0;
#pragma unroll 1
    for(int l = wave*64+lane; l-lane < u.len; l += 256)
    {
        const bool in = l < u.len;
        const double xl = in ? X[l] : 0.0;
#pragma unroll
        for(int h = 0; h < C; h += 16)
            if(u.nc > h)        // uniform, as is every test of nc
            {
                double f[16];
#pragma unroll
                for(int c = 0; c < 16; c++)
                    f[c] = in && h+c < u.nc ? F[(int64_t)(h+c)*u.len+l] : 0.0;
#pragma unroll
                for(int c = 0; c < 16; c++)
                    s[h+c] = fma(f[c], xl, s[h+c]);
            }
    }
    if(u.nc > 16)
    {
        const double t = halving_sum<32>(s, lane);
        if((lane & 1) == 0)
            part[wave][halving_index<32>(lane)] = t;
    }
    else
    {
        double s16[16];
#pragma unroll
        for(int c = 0; c < 16; c++)
            s16[c] = s[c];
        const double t = halving_sum<16>(s16, lane);
        if((lane & 3) == 0)
            part[wave][halving_index<16>(lane)] = t;
    }
    __syncthreads();
    const int c = threadIdx.x;
    if(c < u.nc)
        tmp[u.out_off+c] = ((part[0][c]+part[1][c])+part[2][c])+part[3][c];
}

// The same for up to 16 right-hand sides on MFMA: rows split over the four
// waves in groups of 64, a lane taking rows 4 (lane/16) .. +3 of each block
// of 16 (any order of the rows gives the same sum), so that it loads 32
// contiguous bytes of a column.  Three workgroups per CU: with registers for
// two, N=40000, tile 1265, 7 rhs took 93 instead of 85.5 us.  Lanes past the
// unit's columns or the right-hand sides load column 0 instead of branching
// around the load (only the vectors are set to zero there; the other columns'
// sums are not stored): N=64000, tile 1600, 2 rhs 200 -> 152 us, 16 rhs 716 MB
// 430 -> 303, and the registers allow the four short chains.
__global__ __launch_bounds__(256, 3) void tlr_coef_kernel(
        const tlr_unit *units, const double *fac, const double *x, int ldx,
        int nrhs, double *tmp)
{
    __shared__ double part[3][2][256];
    const tlr_unit u = units[blockIdx.x];
    const int q0 = blockIdx.y*RHS, nq = min(nrhs-q0, RHS);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lc = lane & 15, lr = lane >> 4;
    const double *F[2];
    bool ok[2];
#pragma unroll
    for(int a = 0; a < 2; a++)
    {
        ok[a] = a*16+lc < u.nc;
        F[a] = fac+u.f_off+(int64_t)(ok[a] ? a*16+lc : 0)*u.len;
    }
    const bool okq = lc < nq;
    const double *X = x+u.x_off+(int64_t)(okq ? q0+lc : q0)*ldx;
    Acc<false> acc[2];
    const int nrb = (u.len+15)/16;
    const bool two = u.nc > 16;     // uniform
    for(int g0 = wave*4; g0 < nrb; g0 += 16)
    {
        double f[4][2][4], b[4][4];
        if((g0+4)*16 <= u.len)
        {
            // uniform: a whole group
#pragma unroll
            for(int h = 0; h < 4; h++)
            {
                const int r = (g0+h)*16+4*lr;
#pragma unroll
                for(int v = 0; v < 4; v++)
                {
                    f[h][0][v] = F[0][r+v];
                    b[h][v] = X[r+v];
                }
                if(two)
#pragma unroll
                    for(int v = 0; v < 4; v++)
                        f[h][1][v] = F[1][r+v];
#pragma unroll
                for(int v = 0; v < 4; v++)
                    b[h][v] = okq ? b[h][v] : 0.0;
            }
        }
        else
#pragma unroll
            for(int h = 0; h < 4; h++)
#pragma unroll
                for(int v = 0; v < 4; v++)
                {
                    const int r = (g0+h)*16+4*lr+v;
                    const bool in = r < u.len;
                    f[h][0][v] = in && ok[0] ? F[0][r] : 0.0;
                    f[h][1][v] = in && ok[1] ? F[1][r] : 0.0;
                    b[h][v] = in && okq ? X[r] : 0.0;
                }
        auto sums = [&](int a) {
            Acc<false> p[4];
#pragma unroll
            for(int v = 0; v < 4; v++)
#pragma unroll
                for(int h = 0; h < 4; h++)
                    p[h].add(f[h][a][v], b[h][v]);
            acc[a].v += (p[0].v+p[1].v)+(p[2].v+p[3].v);
        };
        sums(0);
        if(two)
            sums(1);
    }
    if(wave > 0)
#pragma unroll
        for(int a = 0; a < 2; a++)
#pragma unroll
            for(int q = 0; q < 4; q++)
                part[wave-1][a][q*64+lane] = acc[a].v[q];
    __syncthreads();
    if(wave == 0 && okq)
#pragma unroll
        for(int a = 0; a < 2; a++)
#pragma unroll
            for(int q = 0; q < 4; q++)
            {
                const int c = a*16+Acc<false>::row(q, lane);
                if(c < u.nc)
                    tmp[(u.out_off+c)*nrhs+q0+lc] =
                        ((acc[a].v[q]+part[0][a][q*64+lane])+
                         part[1][a][q*64+lane])+part[2][a][q*64+lane];
            }
}

// Rows of a strip of 16 RF rows of one block row.  Up to 32 rows four
// workgroups per CU (with three, N=30000, tile 1100, 3 rhs took 224 instead of
// 212 us).
template <int RF, bool ONE>
__global__ __launch_bounds__(256, RF <= 2 ? 4 : 2) void tlr_rows_kernel(
        const tlr_chunk *chunks, const tlr_entry *entries, const double *fac,
        const double *tmp, const double *x, int ldx, int nrhs, double alpha,
        double beta, double *y, int ldy)
{
    __shared__ double part[3][RF][Acc<ONE>::N*64];
    const tlr_chunk ch = chunks[blockIdx.x];
    const int q0 = blockIdx.y*RHS, nq = min(nrhs-q0, RHS);
    const int lane = threadIdx.x & 63;
    // the wave index as a wave-uniform value: entries are then read through
    // the scalar unit
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lc = lane & 15, lr = lane >> 4;
    const bool okq = ONE || lc < nq;
    const int qx = ONE ? q0 : okq ? q0+lc : q0;
    // rows past the strip repeat its last one (their sums are not stored)
    int row[RF];
#pragma unroll
    for(int a = 0; a < RF; a++)
        row[a] = ch.rofs+min(a*16+lc, ch.nrows-1);
    Acc<ONE> acc[RF], sum[RF];      // of 16 columns, of those before them
    for(int e = ch.first+wave; e < ch.last; e += 4)
    {
        const tlr_entry en = entries[e];
        // element (row, k) of F: kinds 0 and 1 column-major, kind 2 (D^T)
        // row-major
        const bool tr = en.kind == 2;
        const double *F[RF];
#pragma unroll
        for(int a = 0; a < RF; a++)
            F[a] = fac+en.f_off+(tr ? (int64_t)row[a]*en.ld : row[a]);
        const int64_t fs = tr ? 1 : en.ld;
        const double *T = en.kind == 0 ? tmp+en.src_off*nrhs+qx :
            x+en.src_off+(int64_t)qx*ldx;
        const int ts = en.kind == 0 ? nrhs : 1;
        int k0 = 0;
        // a lane's four steps take k = 4 (lane/16) .. +3 of a block of 16
        for(; k0+16 <= en.cols; k0 += 16)
        {
            double f[RF][4], b[4];
#pragma unroll
            for(int a = 0; a < RF; a++)
#pragma unroll
                for(int v = 0; v < 4; v++)
                    f[a][v] = F[a][(k0+4*lr+v)*fs];
#pragma unroll
            for(int v = 0; v < 4; v++)
                b[v] = T[(int64_t)(k0+4*lr+v)*ts];
            if(!ONE)
#pragma unroll
                for(int v = 0; v < 4; v++)
                    b[v] = okq ? b[v] : 0.0;
#pragma unroll
            for(int v = 0; v < 4; v++)
#pragma unroll
                for(int a = 0; a < RF; a++)
                    acc[a].add(f[a][v], b[v]);
#pragma unroll
            for(int a = 0; a < RF; a++)
                sum[a].take(acc[a]);
        }
        if(k0 < en.cols)
        {
            // the last 1-15 columns, loaded together: step v takes
            // k = k0 + 4 v + lane/16
            const int steps = (en.cols-k0+3)/4;     // uniform
            double f[RF][4], b[4];
#pragma unroll
            for(int v = 0; v < 4; v++)
                if(v < steps)
                {
                    const int k = k0+4*v+lr;
                    const bool okk = k < en.cols;
#pragma unroll
                    for(int a = 0; a < RF; a++)
                        f[a][v] = okk ? F[a][k*fs] : 0.0;
                    b[v] = okq && okk ? T[(int64_t)k*ts] : 0.0;
                }
#pragma unroll
            for(int v = 0; v < 4; v++)
                if(v < steps)
#pragma unroll
                    for(int a = 0; a < RF; a++)
                        acc[a].add(f[a][v], b[v]);
#pragma unroll
            for(int a = 0; a < RF; a++)
                sum[a].take(acc[a]);
        }
    }
#pragma unroll
    for(int a = 0; a < RF; a++)
    {
        sum[a].close();
        if(wave > 0)
#pragma unroll
            for(int q = 0; q < Acc<ONE>::N; q++)
                part[wave-1][a][q*64+lane] = sum[a].v[q];
    }
    __syncthreads();
    if(wave == 0 && (ONE ? lane < 16 : okq))
#pragma unroll
        for(int a = 0; a < RF; a++)
#pragma unroll
            for(int q = 0; q < Acc<ONE>::N; q++)
            {
                const int r = a*16+Acc<ONE>::row(q, lane);
                if(r >= ch.nrows)
                    continue;
                const double s = ((sum[a].v[q]+part[0][a][q*64+lane])+
                        part[1][a][q*64+lane])+part[2][a][q*64+lane];
                double *yy = y+(int64_t)(ONE ? q0 : q0+lc)*ldy+ch.row0+r;
                *yy = beta == 0.0 ? alpha*s : fma(alpha, s, beta*(*yy));
            }
}

// Rows of a 64-row strip, one right-hand side: a lane takes a row, so that a
// column is one load of 512 contiguous bytes and its coefficient is the same
// for the whole wave (it comes through the scalar unit).
__global__ __launch_bounds__(256) void tlr_rows1_kernel(
        const tlr_chunk *chunks, const tlr_entry *entries, const double *fac,
        const double *tmp, const double *x, double alpha, double beta,
        double *y)
{
    constexpr int KB = 16;
    __shared__ double part[3][64];
    const tlr_chunk ch = chunks[blockIdx.x];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // rows past the strip repeat its last one (their sums are not stored)
    const int row = ch.rofs+min(lane, ch.nrows-1);
    double sum = 0.0;
    tlr_entry next = {};
    if(ch.first+wave < ch.last)
        next = entries[ch.first+wave];
    for(int e = ch.first+wave; e < ch.last; e += 4)
    {
        const tlr_entry en = next;
        next = entries[min(e+4, ch.last-1)];
        const bool tr = en.kind == 2;
        const double *F = fac+en.f_off+(tr ? (int64_t)row*en.ld : row);
        const int64_t fs = tr ? 1 : en.ld;
        const double *T = (en.kind == 0 ? tmp : x)+en.src_off;
        double s0 = 0.0, s1 = 0.0;
        for(int k0 = 0; k0 < en.cols; k0 += KB)
        {
            const int n = min(en.cols-k0, KB);  // as every test of it, uniform
            double f[KB];
#pragma unroll
            for(int k = 0; k < KB; k += 4)
                if(n >= k+4)
                {
#pragma unroll
                    for(int v = 0; v < 4; v++)
                        f[k+v] = F[(k0+k+v)*fs];
                }
                else
                {
#pragma unroll
                    for(int v = 0; v < 3; v++)
                        if(n > k+v)
                            f[k+v] = F[(k0+k+v)*fs];
                }
#pragma unroll
            for(int k = 0; k < KB; k += 4)
                if(n >= k+4)
                {
#pragma unroll
                    for(int v = 0; v < 4; v += 2)
                    {
                        s0 = fma(f[k+v], T[k0+k+v], s0);
                        s1 = fma(f[k+v+1], T[k0+k+v+1], s1);
                    }
                }
                else
                {
#pragma unroll
                    for(int v = 0; v < 3; v++)
                        if(n > k+v)
                            s0 = fma(f[k+v], T[k0+k+v], s0);
                }
        }
        sum += s0+s1;
    }
    if(wave > 0)
        part[wave-1][lane] = sum;
    __syncthreads();
    if(wave == 0 && lane < ch.nrows)
    {
        const double s = ((sum+part[0][lane])+part[1][lane])+part[2][lane];
        double *yy = y+ch.row0+lane;
        *yy = beta == 0.0 ? alpha*s : fma(alpha, s, beta*(*yy));
    }
}

// ---- vector kernels of conjugate gradients, one column of length n per
// blockIdx.y (columns n apart).  Nothing of an iteration goes to the host:
// the dot products stay as partial sums of at most CG_BLOCKS blocks, which
// every block of the next kernel adds up in the same order, and a column that
// has converged is left alone from then on.

constexpr int CG_BLOCKS = 256;

// Sum of part[0 .. nb) by the whole block (nb <= 256 = blockDim.x), the same
// value in every thread.
__device__ inline double sum_parts(const double *part, int nb)
{
    __shared__ double red[4];
    double s = (int)threadIdx.x < nb ? part[threadIdx.x] : 0.0;
#pragma unroll
    for(int o = 32; o > 0; o >>= 1)
        s += __shfl_xor(s, o, 64);
    if((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = s;
    __syncthreads();
    s = ((red[0]+red[1])+red[2])+red[3];
    __syncthreads();
    return s;
}

__device__ inline void store_part(double s, double *out)
{
    __shared__ double red[4];
#pragma unroll
    for(int o = 32; o > 0; o >>= 1)
        s += __shfl_xor(s, o, 64);
    if((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = s;
    __syncthreads();
    if(threadIdx.x == 0)
        *out = ((red[0]+red[1])+red[2])+red[3];
}

// part[b] = the block's share of a . b
__global__ __launch_bounds__(256) void cg_dot_kernel(const double *a,
        const double *b, int64_t n, double *part)
{
    a += blockIdx.y*n;
    b += blockIdx.y*n;
    double s = 0.0;
    for(int64_t i = (int64_t)blockIdx.x*256+threadIdx.x; i < n;
            i += (int64_t)gridDim.x*256)
        s = fma(a[i], b[i], s);
    store_part(s, part+(int64_t)blockIdx.y*CG_BLOCKS+blockIdx.x);
}

// State of a column before iteration 0 from |r|^2 (cg.c:44-52): the check
// value tol |r_0| and |r_0|^2.
__global__ __launch_bounds__(256) void cg_start_kernel(const double *part,
        int nb, double tol, tlr_cg_state *st)
{
    const double rr = sum_parts(part+(int64_t)blockIdx.x*CG_BLOCKS, nb);
    if(threadIdx.x == 0)
    {
        const double rs = sqrt(rr);
        tlr_cg_state &s = st[blockIdx.x];
        s.rsold = rs*rs;
        s.rscheck = rs*tol;
        s.done = s.rscheck < 0.0 ? -2 : -1;
    }
}

// x += a p, r -= a q with a = rsold/(p . q); part2 = shares of |r|^2
__global__ __launch_bounds__(256) void cg_step_kernel(int64_t n,
        const tlr_cg_state *st, const double *part1, const double *p,
        const double *q, double *x, double *r, double *part2)
{
    const tlr_cg_state s = st[blockIdx.y];
    if(s.done != -1)
        return;
    const int64_t o = blockIdx.y*n;
    const double pq = sum_parts(part1+(int64_t)blockIdx.y*CG_BLOCKS,
            gridDim.x);
    const double a = s.rsold/pq;
    double rr = 0.0;
    for(int64_t i = (int64_t)blockIdx.x*256+threadIdx.x; i < n;
            i += (int64_t)gridDim.x*256)
    {
        x[o+i] = fma(a, p[o+i], x[o+i]);
        const double v = fma(-a, q[o+i], r[o+i]);
        r[o+i] = v;
        rr = fma(v, v, rr);
    }
    store_part(rr, part2+(int64_t)blockIdx.y*CG_BLOCKS+blockIdx.x);
}

// The stopping rule |r| < tol |r_0|, else p = r + |r|^2/rsold p; the new
// state goes to st2 (other blocks still read st).
__global__ __launch_bounds__(256) void cg_next_kernel(int64_t n, int it,
        const tlr_cg_state *st, tlr_cg_state *st2, const double *part2,
        const double *r, double *p)
{
    tlr_cg_state s = st[blockIdx.y];
    if(s.done == -1)
    {
        const double rs = sqrt(sum_parts(part2+(int64_t)blockIdx.y*CG_BLOCKS,
                    gridDim.x));
        if(rs < s.rscheck)
            s.done = it;
        else
        {
            const double b = rs*rs/s.rsold;
            s.rsold = rs*rs;
            const int64_t o = blockIdx.y*n;
            for(int64_t i = (int64_t)blockIdx.x*256+threadIdx.x; i < n;
                    i += (int64_t)gridDim.x*256)
                p[o+i] = fma(b, p[o+i], r[o+i]);
        }
    }
    if(blockIdx.x == 0 && threadIdx.x == 0)
        st2[blockIdx.y] = s;
}

// y = a*x + y
__global__ __launch_bounds__(256) void axpy_kernel(int64_t n, double a,
        const double *x, double *y)
{
    for(int64_t i = (int64_t)blockIdx.x*256+threadIdx.x; i < n;
            i += (int64_t)gridDim.x*256)
        y[i] = fma(a, x[i], y[i]);
}

// y = x
__global__ __launch_bounds__(256) void copy_kernel(int64_t n, const double *x,
        double *y)
{
    for(int64_t i = (int64_t)blockIdx.x*256+threadIdx.x; i < n;
            i += (int64_t)gridDim.x*256)
        y[i] = x[i];
}

inline unsigned vec_grid(int64_t n)
{
    const int64_t g = (n+255)/256;
    return (unsigned)(g < 1024 ? (g > 0 ? g : 1) : 1024);
}

} // namespace


// Scratch of the allocation-free product (starsh_hip_tlr_dmml_noalloc): the
// coefficient blocks V^T X_j and U^T X_i of one call, in a static device
// array that each GPU holds from the load of the library to the end of the
// process.  Host code never uses the array's name as an address: its
// device address is looked up once per device (tlr_scratch_setup, called
// by starsh_hip_init with that device current) and kept in scratch_ptr.
static __device__ __align__(256) double scratch[TLR_SCRATCH_DOUBLES];
static double *scratch_ptr[TLR_MAX_DEVICES];

extern "C" int tlr_scratch_setup(int device)
{
    if(device < 0 || device >= TLR_MAX_DEVICES)
        return STARSH_WRONG_PARAMETER;
    if(scratch_ptr[device] != nullptr)
        return STARSH_SUCCESS;
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if(e != hipSuccess || p == nullptr)
    {
        fprintf(stderr, "STARSH HIP ERROR: hipGetSymbolAddress of the "
                "product scratch failed on device %d: %s\n", device,
                hipGetErrorString(e));
        return STARSH_UNKNOWN_ERROR;
    }
    scratch_ptr[device] = (double *)p;
    return STARSH_SUCCESS;
}

extern "C" int tlr_scratch(int device, double **ptr)
{
    if(device < 0 || device >= TLR_MAX_DEVICES ||
            scratch_ptr[device] == nullptr)
        return STARSH_UNKNOWN_ERROR;
    *ptr = scratch_ptr[device];
    return STARSH_SUCCESS;
}

int starsh_hip_tlr_apply(const tlr_plan *pl, double *d_tmp, int nrhs,
        double alpha, const double *d_x, int ldx, double beta, double *d_y,
        int ldy)
{
    if(nrhs <= 0)
        return STARSH_SUCCESS;
    hipStream_t s = starsh_hip_stream();
    const unsigned groups = (nrhs+RHS-1)/RHS;
    if(pl->nunits > 0)
    {
        if(nrhs == 1)
            hipLaunchKernelGGL(tlr_coef1_kernel, dim3(pl->nunits), dim3(256),
                    0, s, pl->d_units, pl->d_fac, d_x, d_tmp);
        else
            hipLaunchKernelGGL(tlr_coef_kernel, dim3(pl->nunits, groups),
                    dim3(256), 0, s, pl->d_units, pl->d_fac, d_x, ldx, nrhs,
                    d_tmp);
        HIP_TRY(hipGetLastError());
    }
    if(pl->nchunks > 0)
    {
#define ROWS(RF, ONE) hipLaunchKernelGGL((tlr_rows_kernel<RF, ONE>), \
        dim3(pl->nchunks, groups), dim3(256), 0, s, pl->d_chunks, \
        pl->d_entries, pl->d_fac, d_tmp, d_x, ldx, nrhs, alpha, beta, d_y, \
        ldy)
        const bool one = nrhs == 1;
        switch(pl->strip)
        {
            case 16: if(one) ROWS(1, true); else ROWS(1, false); break;
            case 32: if(one) ROWS(2, true); else ROWS(2, false); break;
            case 64:
                if(one && pl->nchunks > ROWS1_STRIPS)
                    hipLaunchKernelGGL(tlr_rows1_kernel, dim3(pl->nchunks),
                            dim3(256), 0, s, pl->d_chunks, pl->d_entries,
                            pl->d_fac, d_tmp, d_x, alpha, beta, d_y);
                else if(one)
                    ROWS(4, true);
                else
                    ROWS(4, false);
                break;
            default: return STARSH_WRONG_PARAMETER;
        }
#undef ROWS
        HIP_TRY(hipGetLastError());
    }
    return STARSH_SUCCESS;
}

static unsigned cg_grid(int64_t n)
{
    const int64_t g = (n+255)/256;
    return (unsigned)(g < CG_BLOCKS ? (g > 0 ? g : 1) : CG_BLOCKS);
}

int starsh_hip_cg_start(int64_t n, int nrhs, double tol, const double *d_r,
        double *d_part, tlr_cg_state *d_st)
{
    const unsigned nb = cg_grid(n);
    for(int q = 0; q < nrhs; q += 65535)
        hipLaunchKernelGGL(cg_dot_kernel, dim3(nb, nrhs-q < 65535 ? nrhs-q :
                    65535), dim3(256), 0, starsh_hip_stream(), d_r+q*n,
                d_r+q*n, n, d_part+(int64_t)q*CG_BLOCKS);
    hipLaunchKernelGGL(cg_start_kernel, dim3(nrhs), dim3(256), 0,
            starsh_hip_stream(), d_part, (int)nb, tol, d_st);
    HIP_TRY(hipGetLastError());
    return STARSH_SUCCESS;
}

int starsh_hip_cg_iteration(int64_t n, int nrhs, int it, double *d_p,
        const double *d_q, double *d_x, double *d_r, double *d_part,
        tlr_cg_state *d_st)
{
    const unsigned nb = cg_grid(n);
    hipStream_t s = starsh_hip_stream();
    for(int q = 0; q < nrhs; q += 65535)
    {
        const unsigned cnt = nrhs-q < 65535 ? nrhs-q : 65535;
        const tlr_cg_state *st = d_st+(int64_t)(it & 1)*nrhs+q;
        tlr_cg_state *st2 = d_st+(int64_t)((it+1) & 1)*nrhs+q;
        double *part1 = d_part+(int64_t)q*CG_BLOCKS;
        double *part2 = part1+(int64_t)nrhs*CG_BLOCKS;
        const int64_t o = q*n;
        hipLaunchKernelGGL(cg_dot_kernel, dim3(nb, cnt), dim3(256), 0, s,
                d_p+o, d_q+o, n, part1);
        hipLaunchKernelGGL(cg_step_kernel, dim3(nb, cnt), dim3(256), 0, s, n,
                st, part1, d_p+o, d_q+o, d_x+o, d_r+o, part2);
        hipLaunchKernelGGL(cg_next_kernel, dim3(nb, cnt), dim3(256), 0, s, n,
                it, st, st2, part2, d_r+o, d_p+o);
    }
    HIP_TRY(hipGetLastError());
    return STARSH_SUCCESS;
}

int starsh_hip_vaxpy(int64_t n, double a, const double *d_x, double *d_y)
{
    hipLaunchKernelGGL(axpy_kernel, dim3(vec_grid(n)), dim3(256), 0,
            starsh_hip_stream(), n, a, d_x, d_y);
    HIP_TRY(hipGetLastError());
    return STARSH_SUCCESS;
}

int starsh_hip_vcopy(int64_t n, const double *d_x, double *d_y)
{
    hipLaunchKernelGGL(copy_kernel, dim3(vec_grid(n)), dim3(256), 0,
            starsh_hip_stream(), n, d_x, d_y);
    HIP_TRY(hipGetLastError());
    return STARSH_SUCCESS;
}

// Seconds per starsh_hip_tlr_apply (mean over reps launches after one
// warm-up), measured with events on the library stream.
int starsh_hip_tlr_time(const tlr_plan *pl, double *d_tmp, int nrhs,
        const double *d_x, int ldx, double *d_y, int ldy, int reps,
        double *seconds)
{
    hipStream_t s = starsh_hip_stream();
    int info = starsh_hip_tlr_apply(pl, d_tmp, nrhs, 1.0, d_x, ldx, 0.0,
            d_y, ldy);
    if(info != STARSH_SUCCESS)
        return info;
    hipEvent_t e0, e1;
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    HIP_TRY(hipEventRecord(e0, s));
    for(int r = 0; r < reps && info == STARSH_SUCCESS; r++)
        info = starsh_hip_tlr_apply(pl, d_tmp, nrhs, 1.0, d_x, ldx, 0.0, d_y,
                ldy);
    HIP_TRY(hipEventRecord(e1, s));
    HIP_TRY(hipEventSynchronize(e1));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *seconds = reps > 0 ? ms*1e-3/reps : 0.0;
    return info;
}

