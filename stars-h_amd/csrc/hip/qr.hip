// Orthogonalisation stages of the randomized SVD: block Gram-Schmidt
// applied twice (BCGS2) with column deflation, compaction of the kept
// columns, and truncation of the projected matrix.
//
// The reference factors the sketch with Householder QR (dgeqrf + dorgqr,
// src/backends/sequential/dense/drsdd.c:64-67).  The sketch of a smooth
// kernel tile is numerically rank deficient far below the sketch width, and
// plain block Gram-Schmidt loses orthogonality on such columns.  Columns
// whose residual after projection falls to tau times their original norm
// are therefore dropped (set to zero): they carry no information above
// rounding, and leaving them out changes the singular values of B = Q^T A
// only at the level of tau*|A|.  Once four columns in a row are dropped, the
// range of the sketch is exhausted and the remaining columns of that tile
// are skipped; a device counter of tiles still in progress lets the host
// stop launching blocks when it reaches zero.
#include "pipeline.h"

namespace {


__device__ inline double wave_sum(double v)
{
    return group_sum_lanes(v, 64);
}

// Column norms squared: which = 0 -> Q buffer (m x k), 2 -> Bt (n x kc).
__global__ __launch_bounds__(256) void colnorm_kernel(const TileDesc *tiles,
        int which, const double *ws, double *out, int kmax)
{
    const TileDesc t = tiles[blockIdx.y];
    const int rows = which == 0 ? t.m : t.n;
    const int cols = which == 0 ? t.k : t.kc;
    const double *base = ws+(which == 0 ? t.q_off : t.bt_off);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for(int c = blockIdx.x*4+wave; c < cols; c += gridDim.x*4)
    {
        const double *col = base+(int64_t)c*rows;
        double s = 0.0;
        for(int i = lane; i < rows; i += 64)
            s += col[i]*col[i];
        s = wave_sum(s);
        if(lane == 0)
            out[(int64_t)blockIdx.y*kmax+c] = s;
    }
}

// ---- Block Gram-Schmidt applied twice (BCGS2)
//
// The columns of Q (which = 0: m rows, width k) or Q2 (which = 1: n rows,
// width p; it starts as Bt[:, :p]) are orthogonalised in blocks of GS_BLOCK.
// For each block, twice:
//   1. C = Q_prev^T W and W -= Q_prev C against the columns before the block
//      (gs_dot_kernel, gs_update_kernel: FP64 MFMA, spread over the chip; C,
//      at most k x 32, in the tile's j_off region, which the core SVD takes
//      over afterwards);
//   2. the block's own columns in panels of PB, one workgroup per tile
//      (gs_inner_kernel): projection against the block's earlier columns,
//      then the panel itself with deflation.  A column whose norm after
//      projection is at most tau times its reference norm (in the first pass
//      the norm of the original column, in the second 1) is set to zero and
//      flagged in keep.
// A tile that drops four columns in a row in the first pass (a whole group,
// starting at a multiple of four) has exhausted its range: the block ends
// there (gs_end), its columns still get the second pass, and later blocks
// are skipped.
//
// The first block takes GS_FIRST columns with no earlier ones, both passes of
// a panel at once, in one launch.
//
// What bounds it: the reads of earlier columns.  A kernel that took one
// 4-column panel per launch through both passes on one workgroup per tile
// re-read every earlier column twice per panel and ran at 4-5 TFLOP/s on
// wide sketches.  A block of 32 re-reads them a quarter as often, on MFMA,
// with as many workgroups as there are 32 x 32 coefficient blocks or 128-row
// strips; panels of 8 instead of 4 columns halve the re-reads inside a
// block.  All launches of one compression on MI355X, before and after: SVD
// engine on 2D exp N=9973 (tile 1000, widths to 1000) 180 -> 16 ms; 3D
// Matern N=65536 (tile 2048, widths to 528) 172 -> 51 ms; 12 exp problems
// (tiles to 2816) 120 -> 32 ms; sin(kr)/r N=25000 (tile 1536, width 400) 39
// -> 9.6 ms; 2D sqexp N=64000 (tile 1600) width 64 2.37 -> 1.85 ms, width 416
// 5.2 -> 3.9 ms.  Widths up to 64 stay in the first block: through the MFMA
// kernels 32 + 32 columns took 2.6 ms there, the block's columns passing
// through HBM once more per launch.
constexpr int GSB = GS_BLOCK;

// Columns of the block at j0.
__host__ __device__ inline int gs_width(int j0)
{
    return j0 == 0 ? GS_FIRST : GSB;
}
static_assert(GSB == 32, "the MFMA kernels below take 32 columns");

typedef double double4_t __attribute__((ext_vector_type(4)));

struct GsView
{
    int rows, width;
    const double *src;     // block W before the first pass
    double *Q;
    bool skip;
};

// pass 0: tiles in progress; pass 1: tiles that took block j0 in pass 0.
__device__ inline GsView gs_view(const TileDesc &t, int which, double *ws,
        int j0, int pass)
{
    GsView v;
    const bool q2 = which != 0;
    v.rows = q2 ? t.n : t.m;
    v.width = q2 ? t.p : t.k;
    v.Q = ws+(q2 ? t.q2_off : t.q_off);
    v.src = (q2 && pass == 0 ? ws+t.bt_off : v.Q)+(int64_t)j0*v.rows;
    v.skip = j0 >= v.width || (pass == 0 ? (t.flags & (q2 ? 2 : 1)) != 0 :
            t.gs_blk != j0 || t.gs_end <= j0);
    return v;
}

// C = Q[:, :j0]^T W, 32 x 32 of it per workgroup, the rows split over its
// four waves; pass 0 also takes the squared norms of W's columns.  Any order
// of the rows gives the same sum, so a lane takes rows 4 (lane/16) .. +3 of
// a 16-row block in its four MFMA steps and loads 32 contiguous bytes.
__global__ __launch_bounds__(256) void gs_dot_kernel(const TileDesc *tiles,
        int which, double *ws, int j0, int pass, double *norms, int kmax)
{
    __shared__ double part[3][16*64];
    __shared__ double npart[4][32];
    const TileDesc &t = tiles[blockIdx.y];
    const GsView g = gs_view(t, which, ws, j0, pass);
    if(g.skip)
        return;
    const int rows = g.rows;
    const int jb = min(g.width-j0, GSB);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lc = lane & 15, lr = lane >> 4;
    const int qc = blockIdx.x*32;
    const double *qa[2], *wb[2];
#pragma unroll
    for(int c = 0; c < 2; c++)
    {
        qa[c] = g.Q+(int64_t)(qc+c*16+lc)*rows;
        wb[c] = g.src+(int64_t)min(c*16+lc, jb-1)*rows;
    }
    const bool want_norm = pass == 0 && blockIdx.x == 0;
    double4_t acc[2][2];
    double sq[2] = {0.0, 0.0};
#pragma unroll
    for(int a = 0; a < 2; a++)
#pragma unroll
        for(int b = 0; b < 2; b++)
            acc[a][b] = double4_t{0.0, 0.0, 0.0, 0.0};
    const int full = rows/16;
    auto step = [&](const double (&fa)[2][4], const double (&fb)[2][4]) {
#pragma unroll
        for(int v = 0; v < 4; v++)
#pragma unroll
            for(int a = 0; a < 2; a++)
#pragma unroll
                for(int b = 0; b < 2; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                            fa[a][v], fb[b][v], acc[a][b], 0, 0, 0);
        if(want_norm)
#pragma unroll
            for(int b = 0; b < 2; b++)
#pragma unroll
                for(int v = 0; v < 4; v++)
                    sq[b] = fma(fb[b][v], fb[b][v], sq[b]);
    };
    for(int rb = wave; rb < full; rb += 4)
    {
        const int r = rb*16+4*lr;
        double fa[2][4], fb[2][4];
#pragma unroll
        for(int c = 0; c < 2; c++)
#pragma unroll
            for(int v = 0; v < 4; v++)
            {
                fa[c][v] = qa[c][r+v];
                fb[c][v] = wb[c][r+v];
            }
        step(fa, fb);
    }
    if(full*16 < rows && (full & 3) == wave)
    {
        const int r = full*16+4*lr;
        double fa[2][4], fb[2][4];
#pragma unroll
        for(int c = 0; c < 2; c++)
#pragma unroll
            for(int v = 0; v < 4; v++)
            {
                fa[c][v] = r+v < rows ? qa[c][r+v] : 0.0;
                fb[c][v] = r+v < rows ? wb[c][r+v] : 0.0;
            }
        step(fa, fb);
    }
    if(wave > 0)
#pragma unroll
        for(int q = 0; q < 16; q++)
            part[wave-1][q*64+lane] = acc[q >> 3][(q >> 2) & 1][q & 3];
    if(want_norm)
    {
#pragma unroll
        for(int b = 0; b < 2; b++)
        {
            sq[b] += __shfl_xor(sq[b], 16, 64);
            sq[b] += __shfl_xor(sq[b], 32, 64);
            if(lr == 0)
                npart[wave][b*16+lc] = sq[b];
        }
    }
    __syncthreads();
    if(wave > 0)
        return;
    double *C = ws+t.j_off;
#pragma unroll
    for(int q = 0; q < 16; q++)
    {
        const int a = q >> 3, b = (q >> 2) & 1, v = q & 3;
        // D layout: row lane/16 + 4 v, column lane%16
        C[(int64_t)(qc+a*16+lr+4*v)*GSB+b*16+lc] = ((acc[a][b][v]+
                part[0][q*64+lane])+part[1][q*64+lane])+part[2][q*64+lane];
    }
    if(want_norm && lane < jb)
        norms[(int64_t)blockIdx.y*kmax+j0+lane] = ((npart[0][lane]+
                npart[1][lane])+npart[2][lane])+npart[3][lane];
}

// W -= Q[:, :j0] C, 128 rows per workgroup, 32 per wave, C (negated) staged
// through LDS 32 rows at a time, double buffered.  Logical row i of a 16-row
// fragment is row 4 (i%4) + i/4 of it, so that a lane's four outputs are
// contiguous.
__global__ __launch_bounds__(256) void gs_update_kernel(
        const TileDesc *tiles, int which, double *ws, int j0, int pass)
{
    __shared__ double Cs[2][32][GSB];
    const TileDesc &t = tiles[blockIdx.y];
    const GsView g = gs_view(t, which, ws, j0, pass);
    const int rows = g.rows;
    if(g.skip || (int)blockIdx.x*128 >= rows)
        return;
    const int jb = min(g.width-j0, GSB);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lc = lane & 15, lr = lane >> 4;
    const int r0 = blockIdx.x*128+wave*32;
    const double *C = ws+t.j_off;
    double4_t acc[2][2];
#pragma unroll
    for(int a = 0; a < 2; a++)
#pragma unroll
        for(int b = 0; b < 2; b++)
#pragma unroll
            for(int v = 0; v < 4; v++)
            {
                const int i = r0+16*a+4*lr+v;
                acc[a][b][v] = i < rows && b*16+lc < jb ?
                    g.src[(int64_t)(b*16+lc)*rows+i] : 0.0;
            }
    const int prow = 4*(lc & 3)+(lc >> 2);
    // rows past the end repeat the last one (their outputs are not stored)
    const double *qr[2];
#pragma unroll
    for(int a = 0; a < 2; a++)
        qr[a] = g.Q+min(r0+16*a+prow, rows-1);
    double creg[4];
#pragma unroll
    for(int e = 0; e < 4; e++)
        creg[e] = C[tid+256*e];
#pragma unroll
    for(int e = 0; e < 4; e++)
        (&Cs[0][0][0])[tid+256*e] = -creg[e];
    __syncthreads();
    int buf = 0;
    for(int k0 = 0; k0 < j0; k0 += 32, buf ^= 1)
    {
        double fa[8][2];
#pragma unroll
        for(int q = 0; q < 8; q++)
#pragma unroll
            for(int a = 0; a < 2; a++)
                fa[q][a] = qr[a][(int64_t)(k0+4*q+lr)*rows];
        const bool more = k0+32 < j0;
        if(more)
#pragma unroll
            for(int e = 0; e < 4; e++)
                creg[e] = C[(int64_t)(k0+32)*GSB+tid+256*e];
#pragma unroll
        for(int q = 0; q < 8; q++)
        {
            const double b0 = Cs[buf][4*q+lr][lc];
            const double b1 = Cs[buf][4*q+lr][16+lc];
#pragma unroll
            for(int a = 0; a < 2; a++)
            {
                acc[a][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[q][a],
                        b0, acc[a][0], 0, 0, 0);
                acc[a][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[q][a],
                        b1, acc[a][1], 0, 0, 0);
            }
        }
        if(more)
#pragma unroll
            for(int e = 0; e < 4; e++)
                (&Cs[buf^1][0][0])[tid+256*e] = -creg[e];
        __syncthreads();
    }
#pragma unroll
    for(int a = 0; a < 2; a++)
#pragma unroll
        for(int b = 0; b < 2; b++)
#pragma unroll
            for(int v = 0; v < 4; v++)
            {
                const int i = r0+16*a+4*lr+v;
                if(i < rows && b*16+lc < jb)
                    g.Q[(int64_t)(j0+b*16+lc)*rows+i] = acc[a][b][v];
            }
}

// The block's own columns (pass `pass`, or both in the first block).  The
// panel lives in registers: thread t
// holds rows t, t+NT, ... (RPT of them), so a thread only ever reads rows
// that it wrote.
template <int NT, int RPT, int PB, int CH>
__global__ __launch_bounds__(NT, 2) void gs_inner_kernel(TileDesc *tiles,
        int which, double *ws, int j0, int pass, int kmax,
        double tau2_first, double tau2_second, int *keep,
        const double *norms, int *active)
{
    constexpr int NW = NT/64, V = CH*PB;
    __shared__ double red[NW][V];
    __shared__ double fin[V];
    __shared__ double pred[2][NW][PB];
    TileDesc &td = tiles[blockIdx.x];
    const GsView g = gs_view(td, which, ws, j0, pass);
    if(g.skip)
        return;
    const bool q2 = which != 0;
    const int rows = g.rows, width = g.width;
    // the first block takes both passes of a panel at once
    const int last = j0 == 0 ? 1 : pass;
    const int end = pass == 0 ? min(j0+gs_width(j0), width) : td.gs_end;
    const bool exhausted_before = (td.flags & (q2 ? 2 : 1)) != 0;
    int *kp = keep+(int64_t)blockIdx.x*kmax;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double *Qb = g.Q;
    // a block with earlier columns was written to Q by the update
    const double *src = (j0 > 0 ? Qb+(int64_t)j0*rows : g.src);
    const int my_idx = halving_index<V>(lane);
    const bool writer = (lane & ((64/V)-1)) == 0;
    int rb = 0;   // partial buffer of the next in-panel reduction
    int stop = end;
    for(int j = j0; j < end; j += PB)
    {
        int jb = end-j < PB ? end-j : PB;
        double *W = Qb+(int64_t)j*rows;
        const double *Wsrc = src+(int64_t)(j-j0)*rows;
        double w[RPT][PB];
#pragma unroll
        for(int r = 0; r < RPT; r++)
        {
            const int i = threadIdx.x+r*NT;
#pragma unroll
            for(int c = 0; c < PB; c++)
                w[r][c] = (i < rows && c < jb) ? Wsrc[(int64_t)c*rows+i] :
                    0.0;
        }
        // deflation reference: squared norms of the original columns
        double ref2[PB];
#pragma unroll
        for(int c = 0; c < PB; c++)
            ref2[c] = pass == 0 && j0 > 0 && c < jb ?
                norms[(int64_t)blockIdx.x*kmax+j+c] : 1.0;
        if(pass == 0 && j0 == 0)
        {
            double v[PB];
#pragma unroll
            for(int c = 0; c < PB; c++)
            {
                double d = 0.0;
#pragma unroll
                for(int r = 0; r < RPT; r++)
                    d += w[r][c]*w[r][c];
                v[c] = d;
            }
            const double tot = halving_sum<PB>(v, lane);
            if((lane & ((64/PB)-1)) == 0)
                red[wave][halving_index<PB>(lane)] = tot;
            __syncthreads();
#pragma unroll
            for(int c = 0; c < PB; c++)
            {
                double sum = 0.0;
#pragma unroll
                for(int q2w = 0; q2w < NW; q2w++)
                    sum += red[q2w][c];
                ref2[c] = sum;
            }
            __syncthreads();
        }
        int cut = PB;
        for(int ps = pass; ps <= last; ps++)
        {
            // ---- projection against the block's columns j0 .. j-1, CH at a
            // time: C = Q_ch^T W, W -= Q_ch C; each chunk of Q is read once,
            // and its CH x PB dot products are reduced by halving_sum, then
            // across the waves in LDS
            for(int l0 = j0; l0 < j; l0 += CH)
            {
                double q[RPT][CH];
#pragma unroll
                for(int r = 0; r < RPT; r++)
                {
                    const int i = threadIdx.x+r*NT;
#pragma unroll
                    for(int c = 0; c < CH; c++)
                        q[r][c] = i < rows ? Qb[(int64_t)(l0+c)*rows+i] : 0.0;
                }
                double v[V];
#pragma unroll
                for(int c = 0; c < CH; c++)
#pragma unroll
                    for(int b = 0; b < PB; b++)
                    {
                        double d = 0.0;
#pragma unroll
                        for(int r = 0; r < RPT; r++)
                            d += q[r][c]*w[r][b];
                        v[c*PB+b] = d;
                    }
                const double tot = halving_sum<V>(v, lane);
                if(writer)
                    red[wave][my_idx] = tot;
                __syncthreads();
                if(threadIdx.x < V)
                {
                    double sum = 0.0;
#pragma unroll
                    for(int q2w = 0; q2w < NW; q2w++)
                        sum += red[q2w][threadIdx.x];
                    fin[threadIdx.x] = sum;
                }
                __syncthreads();
#pragma unroll
                for(int c = 0; c < CH; c++)
#pragma unroll
                    for(int b = 0; b < PB; b++)
                    {
                        const double coef = fin[c*PB+b];
#pragma unroll
                        for(int r = 0; r < RPT; r++)
                            w[r][b] -= q[r][c]*coef;
                    }
            }
            // ---- the panel itself, right-looking with deflation: the
            // products of column c with itself and with the columns after it
            // come from one reduction (one barrier), then column c leaves
            // the later ones.  Once per pass is enough: the second pass
            // starts from columns that are orthogonal up to rounding over
            // tau (max|Q^T Q - I| is 3-6 eps over spectra of eleven orders,
            // steps and cliffs, as with two sweeps in each pass).
            const double tau2 = ps == 0 ? tau2_first : tau2_second;
            int dropped = 0;
#pragma unroll
            for(int c = 0; c < PB; c++)
            {
                if(c < jb && (ps > 0 || cut == PB))
                {
                    double v[PB];
#pragma unroll
                    for(int l = 0; l < PB; l++)
                    {
                        double d = 0.0;
                        if(l >= c)
                        {
#pragma unroll
                            for(int r = 0; r < RPT; r++)
                                d += w[r][l]*w[r][c];
                        }
                        v[l] = d;
                    }
                    const double tot = halving_sum<PB>(v, lane);
                    if((lane & ((64/PB)-1)) == 0)
                        pred[rb][wave][halving_index<PB>(lane)] = tot;
                    __syncthreads();
                    double dot[PB];
#pragma unroll
                    for(int l = 0; l < PB; l++)
                        if(l >= c)
                        {
                            double sum = 0.0;
#pragma unroll
                            for(int q2w = 0; q2w < NW; q2w++)
                                sum += pred[rb][q2w][l];
                            dot[l] = sum;
                        }
                    rb ^= 1;
                    const double n2 = dot[c];
                    const bool drop = !(n2 > tau2*(ps == 0 ? ref2[c] : 1.0)) ||
                        n2 == 0.0;
                    const double inv = drop ? 0.0 : 1.0/sqrt(n2);
#pragma unroll
                    for(int l = 0; l < PB; l++)
                        if(l > c)
                        {
                            const double coef = (dot[l]*inv)*inv;
#pragma unroll
                            for(int r = 0; r < RPT; r++)
                                w[r][l] -= coef*w[r][c];
                        }
#pragma unroll
                    for(int r = 0; r < RPT; r++)
                        w[r][c] *= inv;
                    if(threadIdx.x == 0)
                    {
                        if(ps == 0)
                            kp[j+c] = drop ? 0 : 1;
                        else if(drop)
                            kp[j+c] = 0;
                    }
                    // four columns in a row (from a multiple of four)
                    // dropped: the range is exhausted.  (A selection sketch
                    // A[:, sel] is not a random combination of the columns:
                    // dropped columns do not mean that.)
                    dropped = drop ? dropped+1 : 0;
                    if((c & 3) == 0)
                        dropped = drop ? 1 : 0;
                    if(ps == 0 && ((c & 3) == 3 || c == jb-1) &&
                            dropped == (c & 3)+1 &&
                            !(td.rule & RSDD_RULE_SELECT))
                        cut = c & ~3;
                }
            }
            if(cut < jb)
                jb = cut;
            if(jb == 0)
                break;
        }
#pragma unroll
        for(int r = 0; r < RPT; r++)
        {
            const int i = threadIdx.x+r*NT;
            if(i < rows)
#pragma unroll
                for(int c = 0; c < PB; c++)
                    if(c < jb)
                        W[(int64_t)c*rows+i] = w[r][c];
        }
        if(cut < PB)
        {
            // Q2 is used in place (no compaction): the columns from here on
            // are zeroed and Q2^T Bt ignores them
            stop = j+cut;
            if(q2)
            {
                const int64_t cnt = (int64_t)(width-stop)*rows;
                for(int64_t e = threadIdx.x; e < cnt; e += NT)
                    Qb[(int64_t)stop*rows+e] = 0.0;
            }
            break;
        }
    }
    if(threadIdx.x == 0)
    {
        if(pass == 0)
        {
            td.gs_blk = j0;
            td.gs_end = stop;
            if(stop < end)
            {
                td.flags |= q2 ? 2 : 1;
                atomicSub(active, 1);
            }
        }
        if(last == 1 && end >= width && !exhausted_before && stop == end)
            atomicSub(active, 1);   // finished all blocks
    }
}

// Moves kept columns of Q to the front, in order; sets kc.
__global__ __launch_bounds__(256) void compact_kernel(TileDesc *tiles,
        double *ws, const int *keep, int kmax)
{
    TileDesc &td = tiles[blockIdx.x];
    const int *kp = keep+(int64_t)blockIdx.x*kmax;
    double *Q = ws+td.q_off;
    const int m = td.m;
    int c = 0;
    for(int j = 0; j < td.k; j++)
    {
        if(!kp[j])
            continue;
        if(c != j)
        {
            for(int i = threadIdx.x; i < m; i += blockDim.x)
                Q[(int64_t)c*m+i] = Q[(int64_t)j*m+i];
            __syncthreads();
        }
        c++;
    }
    if(threadIdx.x == 0)
        td.kc = c;
}

// |B|_F^2, truncation point p (smallest p >= 1 whose row tail of B is at
// most (eta*tol)^2 |B|_F^2) and the tail.
__global__ __launch_bounds__(256) void truncate_kernel(TileDesc *tiles,
        int ntiles, const double *bnorm2, int kmax, double eta)
{
    const int t = blockIdx.x*blockDim.x+threadIdx.x;
    if(t >= ntiles)
        return;
    TileDesc &td = tiles[t];
    const double *nb = bnorm2+(int64_t)t*kmax;
    double total = 0.0;
    for(int c = 0; c < td.kc; c++)
        total += nb[c];
    const double eta_tol = eta*td.tol;
    double limit = eta_tol*eta_tol*total;
    int p = td.kc;
    double tail = 0.0;
    while(p > 1 && tail+nb[p-1] <= limit)
    {
        tail += nb[p-1];
        p--;
    }
    if(total == 0.0)
    {
        p = 0;
        tail = 0.0;
    }
    td.p = p;
    td.tail2 = tail;
    td.bnorm2 = total;
}

// Number of tiles that take part in a BCGS2 run (width > 0).
__global__ void count_active_kernel(const TileDesc *tiles, int ntiles,
        int which, int *active)
{
    int c = 0;
    for(int t = threadIdx.x; t < ntiles; t += blockDim.x)
        c += (which ? tiles[t].p : tiles[t].k) > 0;
    for(int o = 32; o > 0; o >>= 1)
        c += __shfl_xor(c, o, 64);
    __shared__ int part[16];
    if((threadIdx.x & 63) == 0)
        part[threadIdx.x >> 6] = c;
    __syncthreads();
    if(threadIdx.x == 0)
    {
        int s = 0;
        for(int q = 0; q < (int)blockDim.x/64; q++)
            s += part[q];
        *active = s;
    }
}

} // namespace

int pipeline_colnorm(const TileDesc *d_tiles, int ntiles, int which,
        double *ws, double *d_norm, int kmax, hipStream_t s)
{
    if(ntiles <= 0)
        return STARSH_SUCCESS;
    int gx = (kmax+3)/4;
    if(gx > 32)
        gx = 32;
    hipLaunchKernelGGL(colnorm_kernel, dim3(gx, ntiles), dim3(256), 0, s,
            d_tiles, which, ws, d_norm, kmax);
    HIP_TRY(hipGetLastError());
    return STARSH_SUCCESS;
}

int pipeline_count_active(const TileDesc *d_tiles, int ntiles, int which,
        int *d_active, hipStream_t s)
{
    hipLaunchKernelGGL(count_active_kernel, dim3(1), dim3(1024), 0, s,
            d_tiles, ntiles, which, d_active);
    HIP_TRY(hipGetLastError());
    return STARSH_SUCCESS;
}

int pipeline_gs_block(TileDesc *d_tiles, int ntiles, int which, double *ws,
        int j0, int pb, int kmax, double tau_first, double tau_second,
        int *d_keep, double *d_norms, int rows_max, int *d_active,
        hipStream_t s)
{
    if(ntiles <= 0)
        return STARSH_SUCCESS;
    for(int pass = 0; pass < (j0 == 0 ? 1 : 2); pass++)
    {
        if(j0 > 0)
        {
            hipLaunchKernelGGL(gs_dot_kernel, dim3(j0/32, ntiles), dim3(256),
                    0, s, d_tiles, which, ws, j0, pass, d_norms, kmax);
            hipLaunchKernelGGL(gs_update_kernel, dim3((rows_max+127)/128,
                        ntiles), dim3(256), 0, s, d_tiles, which, ws, j0,
                    pass);
        }
        // 8-column panels re-read the block's earlier columns half as often
        // as 4-column ones, at the same two tiles per CU; above 2048 rows
        // they do not fit in the registers
#define GS_LAUNCH(NT, RPT, PB, CH) \
        hipLaunchKernelGGL((gs_inner_kernel<NT, RPT, PB, CH>), \
                dim3(ntiles), dim3(NT), 0, s, d_tiles, which, ws, j0, pass, \
                kmax, tau_first*tau_first, tau_second*tau_second, d_keep, \
                d_norms, d_active)
        if(pb == 4 && rows_max <= 1024)
            GS_LAUNCH(256, 4, 4, 4);
        else if(pb == 4 && rows_max <= 2048)
            GS_LAUNCH(256, 8, 4, 4);
        else if(pb == 4 && rows_max <= 4096)
            GS_LAUNCH(512, 8, 4, 4);
        else if(pb == 8 && rows_max <= 1024)
            GS_LAUNCH(256, 4, 8, 4);
        else if(pb == 8 && rows_max <= 2048)
            GS_LAUNCH(256, 8, 8, 2);
#undef GS_LAUNCH
        else
            return STARSH_WRONG_PARAMETER;
        HIP_TRY(hipGetLastError());
    }
    return STARSH_SUCCESS;
}

int pipeline_compact(TileDesc *d_tiles, int ntiles, double *ws,
        const int *d_keep, int kmax, hipStream_t s)
{
    if(ntiles <= 0)
        return STARSH_SUCCESS;
    hipLaunchKernelGGL(compact_kernel, dim3(ntiles), dim3(256), 0, s,
            d_tiles, ws, d_keep, kmax);
    HIP_TRY(hipGetLastError());
    return STARSH_SUCCESS;
}

int pipeline_truncate(TileDesc *d_tiles, int ntiles, double *ws,
        const double *d_bnorm, int kmax, double eta, int nmax,
        hipStream_t s)
{
    (void)nmax;
    if(ntiles <= 0)
        return STARSH_SUCCESS;
    (void)ws;
    hipLaunchKernelGGL(truncate_kernel, dim3((ntiles+255)/256), dim3(256), 0,
            s, d_tiles, ntiles, d_bnorm, kmax, eta);
    HIP_TRY(hipGetLastError());
    return STARSH_SUCCESS;
}
