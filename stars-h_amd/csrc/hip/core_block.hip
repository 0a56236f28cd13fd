// Core SVD of the tiles whose p x p core does not fit in LDS (p >
// CORE_LDS_PMAX, core.hip): one-sided block Jacobi with the work of every
// tile spread over the chip.
//
// The columns of W = R2^T are split into blocks of 16.  A sweep visits every
// pair of blocks once, in rounds of disjoint pairs (circle method), one
// launch per round and one workgroup per block pair and tile:
//   1. Gram matrix G (32 x 32) of the pair's columns on FP64 MFMA;
//   2. one sweep of two-sided Jacobi on G in LDS, all 16 disjoint column
//      pairs of a step at once, the rotations accumulated in J (32 x 32);
//   3. W_pair <- W_pair J on FP64 MFMA (skipped when nothing rotated).
// The rotations and the test |g_ij| > p eps |w_i| |w_j| are those of the
// scalar one-sided method; G is formed afresh from the columns at every
// visit, so its rounding never accumulates, and J is a product of exact-
// to-rounding rotations whose large entries only mix columns of like norm,
// so the small columns of a graded W keep their relative accuracy.  A sweep
// without rotations ends a tile.
//
// What bounds it: a workgroup per tile (the scalar method with column
// blocks in LDS, one rotation per half-wave) left the chip idle below 256
// tiles and paid LDS traffic of O(p) per rotation; here a rotation costs
// O(32) LDS traffic and the O(p) work is MFMA.  A visit is a chain of 31
// steps, each a rotation and two passes through LDS; with 32-column blocks
// (63 steps on 64 x 64 matrices, half the rounds) a round took 118 us instead
// of 35 at p = 150, 130 instead of 44 at 400, 178 instead of 76-82 at 1000
// (four waves), and Matern with 500-row cores was 7% slower as well.  The whole
// 31-step sweep over both blocks' columns converges in about 6 outer sweeps
// where the 16 cross steps alone need 7-8 (numpy model on sin(kr)/r, exp and
// Matern cores).
// Measured on MI355X, all launches of one compression, against one
// workgroup per tile: 2D exp N=9973, tile 1000, SVD engine (10 cores of
// 1000, 45 of 200-500) 1570 -> 22 ms; sin(kr)/r N=25000, tile 1536 (17 of
// 400, 85 of 130-210) 163 -> 6.4 ms; 3D Matern N=65536, tile 2048, mixed
// (up to 528) 191 -> 52 ms.  Only tiles still rotating are launched, by a
// list the sweeps shorten.
#include <float.h>
#include <math.h>
#include "pipeline.h"
#include "jacobi_rotation.h"

typedef double double4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int BW = 16;          // columns per block
constexpr int PW = 2*BW;        // columns per block pair
constexpr int NT = 256;         // threads of a round: 4 waves
constexpr int OB = 32;          // columns per block of jb_off_kernel

__device__ inline int ld_of(int p)
{
    return (p+15)/16*16;
}

// Number of column blocks, rounded up to even (the last may be empty).
__host__ __device__ inline int blocks_of(int p)
{
    const int nb = (p+BW-1)/BW;
    return nb+(nb & 1);
}

// Largest entry of R2, kept in td.off2 until the first sweep is over, as the
// bit pattern of a non-negative double (they order like integers); one
// workgroup per 8 columns.
__global__ __launch_bounds__(256) void jb_max_kernel(TileDesc *tiles,
        const int *list, const double *ws)
{
    TileDesc &td = tiles[list[blockIdx.y]];
    const int p = td.p, k = td.k;
    const double *R2 = ws+td.r_off;
    double v = 0.0;
    // R2 is upper triangular up to rounding, but every entry is taken
    const int c1 = min(p, (int)blockIdx.x*8+8);
    for(int c = blockIdx.x*8+(threadIdx.x >> 6); c < c1; c += 4)
        for(int i = threadIdx.x & 63; i < p; i += 64)
            v = fmax(v, fabs(R2[(int64_t)c*k+i]));
    for(int o = 32; o > 0; o >>= 1)
        v = fmax(v, __shfl_xor(v, o, 64));
    if((threadIdx.x & 63) == 0)
        atomicMax((unsigned long long *)&td.off2,
                (unsigned long long)__double_as_longlong(v));
}

// Exponent of the scale of W.
__device__ inline int scale_exponent(const TileDesc &td)
{
    const double wm = td.off2;
    int e = 0;
    if(wm > 0.0 && wm < INFINITY)
        frexp(wm, &e);
    return e;
}

// The start of the tiles' Jacobi state.
__global__ __launch_bounds__(256) void jb_state_kernel(TileDesc *tiles,
        const int *list, int count)
{
    const int t = blockIdx.x*256+threadIdx.x;
    if(t >= count)
        return;
    TileDesc &td = tiles[list[t]];
    td.jrot = 0;
    td.jdone = 0;
    td.sweeps = 0;
    td.off2 = 0.0;
}

// W = R2^T 2^-wexp (the power of two that brings the largest entry into
// [1/2, 1), exact), rows padded to 16 and columns to 64 with zeros: zero
// columns never rotate.  One 32 x 32 patch per workgroup, transposed in
// LDS.
__global__ __launch_bounds__(256) void jb_init_kernel(TileDesc *tiles,
        const int *list, double *ws)
{
    TileDesc &td = tiles[list[blockIdx.y]];
    const int p = td.p, k = td.k;
    const int ld = ld_of(p), nc = (p+63)/64*64;
    const int pr = (ld+31)/32;
    const int bi = blockIdx.x % pr, bj = blockIdx.x / pr;
    if(bj*32 >= nc)
        return;
    const double *R2 = ws+td.r_off;
    double *W = ws+td.j_off;
    const int wexp = scale_exponent(td);
    const double scale = ldexp(1.0, -wexp);
    if(blockIdx.x == 0 && threadIdx.x == 0)
        td.wexp = wexp;
    __shared__ double patch[32][33];
    const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
    // W(i, j) = R2(j, i): column i of R2 is read along j
    for(int r = y; r < 32; r += 8)
    {
        const int i = bi*32+r, j = bj*32+x;
        patch[r][x] = i < p && j < p ? R2[(int64_t)i*k+j]*scale : 0.0;
    }
    __syncthreads();
    for(int r = y; r < 32; r += 8)
    {
        const int i = bi*32+x, j = bj*32+r;
        if(i < ld)
            W[(int64_t)j*ld+i] = patch[x][r];
    }
}

// Column at position x of the circle method at a step (position 0 is fixed).
__device__ inline int column_of(int x, int step)
{
    int c = x+step;
    c = c > PW-1 ? c-(PW-1) : c;
    return x == 0 ? 0 : c;
}

// One round of a sweep: workgroup (x, y) handles pair x of the circle method
// on the column blocks of tile list[y].
__global__ __launch_bounds__(NT) void jb_round_kernel(TileDesc *tiles,
        const int *list, double *ws, int round)
{
    __shared__ double G[PW*PW];
    __shared__ double J[PW*PW];
    __shared__ double part[2][3*256];
    __shared__ double2 cs[NT/64][BW];
    __shared__ int perm[PW];
    if(list[blockIdx.y] < 0)
        return;
    TileDesc &td = tiles[list[blockIdx.y]];
    const int p = td.p;
    if(td.jdone)
        return;
    const int nbe = blocks_of(p);
    const int x = blockIdx.x, y = nbe-1-x;
    if(round >= nbe-1 || x >= nbe/2)
        return;
    const int bi = x == 0 ? 0 : 1+(x-1+round) % (nbe-1);
    const int bj = 1+(y-1+round) % (nbe-1);
    const int ld = ld_of(p);
    double *W = ws+td.j_off;
    double *WI = W+(int64_t)bi*BW*ld, *WJ = W+(int64_t)bj*BW*ld;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lc = lane & 15, lr = lane >> 4;
    const int nrb = ld/16;

    // ---- 1. G = [WI WJ]^T [WI WJ], rows split over the waves in blocks of
    // 16.  A and B operand have the same layout (lane: column lane%16, row
    // lane/16 of a step); any order of the rows gives the same sum, so a
    // lane takes rows 4 (lane/16) .. +3 of the block in its four steps and
    // loads 32 contiguous bytes.
    double4_t gii = {0.0, 0.0, 0.0, 0.0}, gij = gii, gjj = gii;
    for(int r0 = wave; r0 < nrb; r0 += 4)
    {
        const int64_t o = (int64_t)lc*ld+r0*16+4*lr;
        double fi[4], fj[4];
#pragma unroll
        for(int v = 0; v < 4; v++)
        {
            fi[v] = WI[o+v];
            fj[v] = WJ[o+v];
        }
#pragma unroll
        for(int v = 0; v < 4; v++)
        {
            gii = __builtin_amdgcn_mfma_f64_16x16x4f64(fi[v], fi[v], gii,
                    0, 0, 0);
            gij = __builtin_amdgcn_mfma_f64_16x16x4f64(fi[v], fj[v], gij,
                    0, 0, 0);
            gjj = __builtin_amdgcn_mfma_f64_16x16x4f64(fj[v], fj[v], gjj,
                    0, 0, 0);
        }
    }
    // sum over the waves in a fixed order, halving their number
#pragma unroll
    for(int h = 2; h > 0; h >>= 1)
    {
        if(wave >= h && wave < 2*h)
#pragma unroll
            for(int v = 0; v < 4; v++)
            {
                part[wave-h][v*64+lane] = gii[v];
                part[wave-h][256+v*64+lane] = gij[v];
                part[wave-h][512+v*64+lane] = gjj[v];
            }
        __syncthreads();
        if(wave < h)
#pragma unroll
            for(int v = 0; v < 4; v++)
            {
                gii[v] += part[wave][v*64+lane];
                gij[v] += part[wave][256+v*64+lane];
                gjj[v] += part[wave][512+v*64+lane];
            }
        __syncthreads();
    }
    if(wave == 0)
    {
        // D layout: row lane/16 + 4 v, column lane%16
#pragma unroll
        for(int v = 0; v < 4; v++)
        {
            const int i = lr+4*v;
            G[i*PW+lc] = gii[v];
            G[i*PW+16+lc] = gij[v];
            G[(16+lc)*PW+i] = gij[v];
            G[(16+i)*PW+16+lc] = gjj[v];
        }
    }
    for(int e = threadIdx.x; e < PW*PW; e += NT)
        J[e] = e % PW == e/PW ? 1.0 : 0.0;
    __syncthreads();

    // most visits of the last sweeps have nothing to rotate: all pairs are
    // tested at once first
    const double ctol = (double)p*DBL_EPSILON;
    {
        bool any = false;
        for(int e = threadIdx.x; e < PW*PW; e += NT)
        {
            const int i = e/PW, j = e % PW;
            if(i < j)
                any |= jr_rotates(G[i*(PW+1)], G[j*(PW+1)], G[e], ctol);
        }
        if(__syncthreads_or(any) == 0)
            return;
    }

    // ---- 2. one sweep of Jacobi on G.  Lane l of every wave computes the
    // rotation of column pair l%16 of the step (so the step needs no
    // exchange of rotations between waves); the 16 lane groups of the
    // workgroup take a row pair of G (2 x 2 blocks with column pair l%16) and
    // two rows of J.  J is one step behind, so that its LDS traffic overlaps
    // the latency of the next rotations.
    const int pj = lane & 15;
    const int slot = wave*4+lr;
    bool rotated = false;
    double pc = 1.0, ps = 0.0;          // rotation J has not seen yet
    int pa = 0, pb = 1;
    auto rotate_j = [&]() {
#pragma unroll
        for(int q = 0; q < 2; q++)
        {
            double *row = J+(q*16+slot)*PW;
            const double u = row[pa], v = row[pb];
            row[pa] = pc*u-ps*v;
            row[pb] = ps*u+pc*v;
        }
    };
    for(int step = 0; step < PW-1; step++)
    {
        const int ca = column_of(pj, step), cb = column_of(PW-1-pj, step);
        const double al = G[ca*PW+ca], be = G[cb*PW+cb];
        const double ga = G[ca*PW+cb];
        rotate_j();
        pc = 1.0;
        ps = 0.0;
        double c = 1.0, s = 0.0;
        const bool rot = jr_rotates(al, be, ga, ctol);
        if(rot)
            jacobi_rotation(al, be, ga, c, s);
        if(__ballot(rot) == 0)
            continue;               // the same in every wave
        rotated = true;
        // the rotations of the step for the rows (each wave its own copy)
        if(lane < BW)
            cs[wave][pj] = double2{c, s};
        // every wave has read its rotations before G changes
        __syncthreads();
        // G <- R^T G R
        const int ra = column_of(slot, step);
        const int rb = column_of(PW-1-slot, step);
        const double ci = cs[wave][slot].x, si = cs[wave][slot].y;
        const double gaa = G[ra*PW+ca], gab = G[ra*PW+cb];
        const double gba = G[rb*PW+ca], gbb = G[rb*PW+cb];
        const double xaa = c*gaa-s*gab, xab = s*gaa+c*gab;
        const double xba = c*gba-s*gbb, xbb = s*gba+c*gbb;
        G[ra*PW+ca] = ci*xaa-si*xba;
        G[ra*PW+cb] = ci*xab-si*xbb;
        G[rb*PW+ca] = si*xaa+ci*xba;
        G[rb*PW+cb] = si*xab+ci*xbb;
        pc = c;
        ps = s;
        pa = ca;
        pb = cb;
        __syncthreads();
    }
    if(!rotated)
        return;
    rotate_j();
    if(threadIdx.x == 0)
        atomicAdd(&td.jrot, 1);
    // the columns leave sorted by norm, the larger ones to the first block:
    // clusters of nearly equal singular values (a diagonal tile of points
    // on equal spheres) converge in 14-16 sweeps sorted and 26 unsorted
    if(threadIdx.x < PW)
    {
        const double v = G[threadIdx.x*(PW+1)];
        int pos = 0;
        for(int l = 0; l < PW; l++)
        {
            const double o = G[l*(PW+1)];
            pos += o > v || (o == v && l < (int)threadIdx.x);
        }
        perm[bi < bj ? pos : pos^BW] = threadIdx.x;
    }
    __syncthreads();

    // ---- 3. W_pair <- W_pair J, rows split over the waves in blocks of 16;
    // a wave reads a block's rows before it writes them.  Logical row i of
    // the block is physical row 4 (i%4) + i/4, so that the output lane stores
    // 4 consecutive rows.
    double jb[8][2];
#pragma unroll
    for(int q = 0; q < 8; q++)
#pragma unroll
        for(int n = 0; n < 2; n++)
            jb[q][n] = J[(4*q+lr)*PW+perm[16*n+lc]];
    const int prow = 4*(lc & 3)+(lc >> 2);
    for(int r0 = wave; r0 < nrb; r0 += 4)
    {
        double a[8];
#pragma unroll
        for(int q = 0; q < 8; q++)
            a[q] = (q < 4 ? WI : WJ)[(int64_t)(4*(q & 3)+lr)*ld+r0*16+prow];
        double4_t acc[2];
#pragma unroll
        for(int n = 0; n < 2; n++)
            acc[n] = double4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for(int q = 0; q < 8; q++)
#pragma unroll
            for(int n = 0; n < 2; n++)
                acc[n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], jb[q][n],
                        acc[n], 0, 0, 0);
#pragma unroll
        for(int n = 0; n < 2; n++)
        {
            double *dst = (n == 0 ? WI : WJ)+(int64_t)lc*ld+r0*16+4*lr;
#pragma unroll
            for(int v = 0; v < 4; v++)
                dst[v] = acc[n][v];
        }
    }
}

// Whether the tile may end with the verdict "rank above the limit" alone
// (its singular values are not asked for), and that limit.
__device__ inline bool rank_limit(const TileDesc &td, int &limit)
{
    const int mn = td.m < td.n ? td.m : td.n;
    limit = td.maxrank;
    if((td.rule & RSDD_RULE_HALF) && mn/2-1 < limit)
        limit = mn/2-1;
    return td.nosv && !td.jdone && td.p > limit;
}

// Squared norms of W's columns (to the tile's S) and the sum of the squares
// of the Gram matrix's strict upper triangle (td.off2): one workgroup per
// block pair I <= J.
__global__ __launch_bounds__(256) void jb_off_kernel(TileDesc *tiles,
        const int *list, double *ws)
{
    __shared__ double part[3][16*64];
    if(list[blockIdx.y] < 0)
        return;
    TileDesc &td = tiles[list[blockIdx.y]];
    int limit;
    if(!rank_limit(td, limit))
        return;
    const int p = td.p, nb = (p+OB-1)/OB;
    int bi = 0, rest = blockIdx.x;
    while(bi < nb && rest >= nb-bi)
        rest -= nb-bi++;
    if(bi >= nb)
        return;
    const int bj = bi+rest, ld = ld_of(p);
    const double *WI = ws+td.j_off+(int64_t)bi*OB*ld;
    const double *WJ = ws+td.j_off+(int64_t)bj*OB*ld;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lc = lane & 15, lr = lane >> 4;
    double4_t g[2][2];
#pragma unroll
    for(int a = 0; a < 2; a++)
#pragma unroll
        for(int b = 0; b < 2; b++)
            g[a][b] = double4_t{0.0, 0.0, 0.0, 0.0};
    for(int rb = wave; rb < ld/16; rb += 4)
#pragma unroll
        for(int v = 0; v < 4; v++)
        {
            double fa[2], fb[2];
#pragma unroll
            for(int c = 0; c < 2; c++)
            {
                fa[c] = WI[(int64_t)(c*16+lc)*ld+rb*16+4*lr+v];
                fb[c] = WJ[(int64_t)(c*16+lc)*ld+rb*16+4*lr+v];
            }
#pragma unroll
            for(int a = 0; a < 2; a++)
#pragma unroll
                for(int b = 0; b < 2; b++)
                    g[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[a],
                            fb[b], g[a][b], 0, 0, 0);
        }
    if(wave > 0)
#pragma unroll
        for(int t = 0; t < 16; t++)
            part[wave-1][t*64+lane] = g[t >> 3][(t >> 2) & 1][t & 3];
    __syncthreads();
    if(wave > 0)
        return;
    double off = 0.0;
#pragma unroll
    for(int t = 0; t < 16; t++)
    {
        const int a = t >> 3, b = (t >> 2) & 1, v = t & 3;
        const double x = ((g[a][b][v]+part[0][t*64+lane])+
                part[1][t*64+lane])+part[2][t*64+lane];
        const int i = bi*OB+a*16+lr+4*v, j = bj*OB+b*16+lc;
        if(i < j)
            off += x*x;
        else if(i == j && i < p)
            ws[td.s_off+i] = x;
    }
    for(int o = 32; o > 0; o >>= 1)
        off += __shfl_xor(off, o, 64);
    if(lane == 0)
        atomicAdd(&td.off2, off);
}

// Ends the tiles whose rank is certainly above the limit.  With d the
// squared column norms of W in descending order and E the off-diagonal part
// of W^T W, Hoffman and Wielandt's theorem gives sum |lambda_i - d_i|^2 <=
// |E|_F^2, so the energy past the limit, sum_{i > limit} lambda_i, is at
// least sum_{i > limit} d_i - sqrt(p - limit) |E|_F.  Twice the energy that
// the rank rule allows (tol^2 of the total) is asked for, far more than any
// rounding, so the verdict is the one the converged singular values give.
__global__ __launch_bounds__(256) void jb_cert_kernel(TileDesc *tiles,
        const int *list, const double *ws)
{
    __shared__ double d[1024];
    __shared__ double part[2][4];
    if(list[blockIdx.x] < 0)
        return;
    TileDesc &td = tiles[list[blockIdx.x]];
    int limit;
    if(!rank_limit(td, limit))
        return;
    const int p = td.p;
    for(int i = threadIdx.x; i < p; i += 256)
        d[i] = ws[td.s_off+i];
    __syncthreads();
    double tail = 0.0, total = 0.0;
    for(int i = threadIdx.x; i < p; i += 256)
    {
        const double v = d[i];
        int pos = 0;
        for(int l = 0; l < p; l++)
            pos += d[l] > v || (d[l] == v && l < i);
        total += v;
        if(pos >= limit)
            tail += v;
    }
    for(int o = 32; o > 0; o >>= 1)
    {
        tail += __shfl_xor(tail, o, 64);
        total += __shfl_xor(total, o, 64);
    }
    if((threadIdx.x & 63) == 0)
    {
        part[0][threadIdx.x >> 6] = tail;
        part[1][threadIdx.x >> 6] = total;
    }
    __syncthreads();
    if(threadIdx.x == 0)
    {
        const double t2 = ldexp(td.tail2, -2*td.wexp);
        tail = part[0][0]+part[0][1]+part[0][2]+part[0][3]+t2;
        total = part[1][0]+part[1][1]+part[1][2]+part[1][3]+t2;
        const double low = tail-sqrt(2.0*td.off2*(p-limit));
        if(low > 2.0*td.tol*td.tol*total && low > 1e-12*total)
            td.jdone = 2;
        td.off2 = 0.0;
    }
}

// End of a sweep: tiles without a rotation are done; the others stay on the
// list, in order, followed by -1.  out[0] = their number, out[1] = the largest
// of their p.
__global__ __launch_bounds__(1024) void jb_sweep_kernel(TileDesc *tiles,
        int *list, int count, int *out)
{
    __shared__ int wcount[16], wmax[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int base = 0, pmax = 0;
    for(int c0 = 0; c0 < count; c0 += 1024)
    {
        const int q = c0+threadIdx.x;
        bool keep = false;
        int t = 0, p = 0;
        if(q < count && (t = list[q]) >= 0)
        {
            TileDesc &td = tiles[t];
            if(!td.jdone)
            {
                if(td.jrot == 0)
                    td.jdone = 1;
                else
                {
                    td.sweeps++;
                    td.jrot = 0;
                    td.off2 = 0.0;
                    keep = true;
                    p = td.p;
                }
            }
        }
        const unsigned long long m = __ballot(keep);
        for(int o = 32; o > 0; o >>= 1)
            p = max(p, __shfl_xor(p, o, 64));
        if(lane == 0)
        {
            wcount[wave] = __popcll(m);
            wmax[wave] = p;
        }
        __syncthreads();
        int before = base;
        for(int w = 0; w < 16; w++)
        {
            before += w < wave ? wcount[w] : 0;
            base += wcount[w];
            pmax = max(pmax, wmax[w]);
        }
        // places before q only: an entry read later is never overwritten
        if(keep)
            list[before+__popcll(m & ((1ull << lane)-1))] = t;
        __syncthreads();
    }
    for(int q = base+threadIdx.x; q < count; q += 1024)
        list[q] = -1;
    if(threadIdx.x == 0)
    {
        out[0] = base;
        out[1] = pmax;
    }
}

} // namespace

// Jacobi sweeps on the count tiles of d_list (the tiles with a core beyond
// LDS; the list is used up): W (columns orthogonal on return) in the tile's
// j_off region, ld = p rounded up to 16, scaled by 2^-wexp, td.jdone 1; tiles
// that ended early with a rank certainly above the limit have jdone 2, tiles
// that did not converge 0.  certify: some tile may end that way.  d_out: two
// device ints, h_out: two pinned host ints.
int pipeline_jacobi_block(TileDesc *d_tiles, int *d_list, int count,
        double *ws, int pmax, int max_sweeps, bool certify, int *d_out,
        int *h_out, hipStream_t s)
{
    if(count <= 0)
        return STARSH_SUCCESS;
    hipLaunchKernelGGL(jb_state_kernel, dim3((count+255)/256), dim3(256), 0,
            s, d_tiles, d_list, count);
    hipLaunchKernelGGL(jb_max_kernel, dim3((pmax+7)/8, count), dim3(256), 0,
            s, d_tiles, d_list, ws);
    hipLaunchKernelGGL(jb_init_kernel, dim3((pmax+31)/32*
                ((pmax+63)/64*2), count),
            dim3(256), 0, s, d_tiles, d_list, ws);
    HIP_TRY(hipGetLastError());
    for(int sweep = 0; sweep < max_sweeps; sweep++)
    {
        const int nbe = blocks_of(pmax);
        for(int round = 0; round < nbe-1; round++)
            hipLaunchKernelGGL(jb_round_kernel, dim3(nbe/2, count), dim3(NT),
                    0, s, d_tiles, d_list, ws, round);
        // Tiles headed for a rank above the limit are tried after sweeps 3
        // to 7, a try being 7-8% of a sweep.  Of those that end so, sin(kr)/r
        // (17 tiles of 400) loses 16 after sweep 4, the SVD engine on 2D exp
        // (10 of 1000) 4 after 3 and 6 after 4, 56 tiles of 12 exp problems
        // (400) and 32 of 3D Matern (528) more by 5 to 7; after sweep 2 it
        // was one of 248.  Device time without any try, with tries after 2,
        // 3, 4 and 7, and so: 50.9, 35.8, 35.8 ms; 79.1, 47.1, 46.6; 84.5,
        // 83, 80.5; 229, 227, 225.
        if(certify && sweep >= 2 && sweep <= 6)
        {
            const int nb = (pmax+OB-1)/OB;
            hipLaunchKernelGGL(jb_off_kernel, dim3(nb*(nb+1)/2, count),
                    dim3(256), 0, s, d_tiles, d_list, ws);
            hipLaunchKernelGGL(jb_cert_kernel, dim3(count), dim3(256), 0, s,
                    d_tiles, d_list, ws);
        }
        hipLaunchKernelGGL(jb_sweep_kernel, dim3(1), dim3(1024), 0, s,
                d_tiles, d_list, count, d_out);
        HIP_TRY(hipGetLastError());
        // no core of this size converges in two sweeps unless it was
        // diagonal from the start
        if(sweep < 1)
            continue;
        HIP_TRY(hipMemcpyAsync(h_out, d_out, 2*sizeof(int),
                    hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        count = h_out[0];
        if(count == 0)
            break;
        pmax = h_out[1];
    }
    return STARSH_SUCCESS;
}
